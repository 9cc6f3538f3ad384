"""The staged integer products (csrc/gemm_i8.hip): sizes at the edges of its tiles and stages, rows of every alignment, zero
points, transposed and strided operands, against exact sums in float64 on rows at the edges of the tiles."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# M, K, N and the tile that the rule takes with b as it is and transposed (None: another kernel); K: whole stages, one more, one less, none whole
SHAPES = [
    (1024, 1024, 4096, "2, 2, 2", "2, 2, 2"), (1100, 1025, 2500, "2, 2, 2", "2, 2, 2"), (2049, 895, 3050, "1, 2, 4", "2, 2, 2"), (2051, 1024, 1025, "2, 2, 2", "2, 2, 2"), (1500, 389, 5000, "2, 2, 2", "2, 2, 2"),
    (512, 1024, 4096, "1, 2, 4", "1, 2, 4"), (900, 513, 2050, "1, 2, 4", "1, 2, 4"), (1100, 700, 1505, "1, 2, 4", "1, 2, 4"),
    (130, 4096, 4096, "1, 1, 8", "1, 1, 8"), (63, 4001, 4099, "1, 1, 8", "1, 1, 8"), (577, 1537, 835, "1, 1, 8", "1, 1, 8"), (4099, 2303, 65, "1, 1, 8", "1, 1, 8"),
    (64, 2048, 16, None, None), (600, 190, 900, None, None),
]


@pytest.fixture(scope="module")
def g():
    import gpu_util
    return gpu_util


def codes(rng, shape, dt):
    lo, hi = (0, 256) if dt == np.uint8 else (-128, 128)
    return rng.integers(lo, hi, size=shape).astype(dt)


def rows_of(M):
    return sorted({r for r in (0, 1, 31, 32, 63, 64, 127, 128, M - 2, M - 1) if r < M})


@pytest.mark.parametrize("M,K,N,tile,tile_transposed", SHAPES)
@pytest.mark.parametrize("dts", [(np.uint8, np.int8), (np.int8, np.uint8)])
def test_matmul_integer(g, M, K, N, tile, tile_transposed, dts):
    rng = np.random.default_rng(M + K + N)
    a, b = codes(rng, (M, K), dts[0]), codes(rng, (K, N), dts[1])
    rows = rows_of(M)
    a64, b64 = a[rows].astype(np.float64), b.astype(np.float64)
    apart = torch.zeros((M, K + 21), dtype=g.dev(a[:1]).dtype, device="cuda")  # rows further apart than they are long
    apart[:, 5:5 + K] = g.dev(a)
    bt = g.dev(np.ascontiguousarray(b.T)).t()
    for az, bz in [(128 if dts[0] == np.uint8 else 0, np.asarray(0 if dts[1] == np.int8 else 128)), (7, rng.integers(0, 100, size=N))]:
        want = np.matmul(a64 - az, b64 - bz).astype(np.int64).astype(np.int32)  # (exact: below 2^53)
        azt, bzt = g.dev(np.asarray(az).astype(dts[0])), g.dev(bz.astype(dts[1]))
        for x, y in [(g.dev(a), g.dev(b)), (apart[:, 5:5 + K], g.dev(b)), (g.dev(a), bt)]:
            got = g.ops.MatMulInteger(x, y, azt, bzt)
            np.testing.assert_array_equal(g.host(got)[rows], want)
        # every row, against itself in another order
        flip = g.ops.MatMulInteger(g.dev(np.ascontiguousarray(a[::-1])), g.dev(b), azt, bzt)
        assert torch.equal(flip.flip(0), got)


@pytest.mark.parametrize("M,K,N,tile,tile_transposed", SHAPES)
def test_qlinear_matmul(g, oracle, M, K, N, tile, tile_transposed):
    rng = np.random.default_rng(M + K)
    a, b, bias = codes(rng, (M, K), np.uint8), codes(rng, (K, N), np.int8), rng.integers(-3000, 3000, size=N).astype(np.int32)
    rows, s_y = rows_of(M), float(0.02 * 0.005 * 74 * 74 * np.sqrt(K) / 32)
    bt = g.dev(np.ascontiguousarray(b.T)).t()
    for bz, rne in [(0, False), (4, True)]:
        fl = g.capi.ROUND_ONNX_RNE if rne else 0
        want = oracle.qlinear_matmul_int(a[rows], 0.02, 117, b, 0.005, bz, s_y, 128, bias=bias, round_mode=oracle.ROUND_ONNX_RNE if rne else oracle.ROUND_REFERENCE)
        for y in (g.dev(b), bt):
            got = g.host(g.ops.QLinearMatMul(g.dev(a), 0.02, 117, y, 0.005, bz, s_y, 128, g.dev(bias), flags=fl))
            np.testing.assert_array_equal(got[rows], want)


def test_batches(g):
    rng = np.random.default_rng(3)
    a, b = codes(rng, (3, 300, 1030), np.uint8), codes(rng, (3, 1030, 1300), np.int8)
    got = g.host(g.ops.MatMulInteger(g.dev(a), g.dev(b), g.dev(np.array(9, np.uint8)), g.dev(np.array(-5, np.int8))))
    want = np.matmul(a[:, ::37].astype(np.float64) - 9, b.astype(np.float64) + 5).astype(np.int32)
    np.testing.assert_array_equal(got[:, ::37], want)


# rows of b of 4 to 15 bytes, whole stages of 128 and a rest; rows next to each other, 9 bytes apart, b transposed (1)
@pytest.mark.parametrize("M,K,N", [(65300, 768, 4), (65281, 1023, 15), (65408, 1280, 10), (65285, 897, 7)])
@pytest.mark.parametrize("apart", [0, 1, 9])
def test_few_columns(g, oracle, M, K, N, apart):
    rng = np.random.default_rng(K + N + apart)
    a, b = codes(rng, (M, K), np.uint8), codes(rng, (K, N), np.int8)
    rows = rows_of(M)
    bd = torch.zeros(K * (N + apart) - apart, dtype=torch.int8, device="cuda").as_strided((K, N), (N + apart, 1))  # ends with its last element
    bd.copy_(g.dev(b))
    if apart == 1:
        bd = g.dev(np.ascontiguousarray(b.T)).t()
    for az, bz in [(128, np.asarray(0)), (7, rng.integers(-90, 90, size=N))]:
        got = g.ops.MatMulInteger(g.dev(a), bd, g.dev(np.asarray(az, np.uint8)), g.dev(bz.astype(np.int8)))
        want = np.matmul(a[rows].astype(np.float64) - az, b.astype(np.float64) - bz).astype(np.int64).astype(np.int32)  # (exact: below 2^53)
        np.testing.assert_array_equal(g.host(got)[rows], want)
        flip = g.ops.MatMulInteger(g.dev(np.ascontiguousarray(a[::-1])), bd, g.dev(np.asarray(az, np.uint8)), g.dev(bz.astype(np.int8)))
        assert torch.equal(flip.flip(0), got)
    bias, s_y = rng.integers(-3000, 3000, size=N).astype(np.int32), float(0.02 * 0.005 * 74 * 74 * np.sqrt(K) / 32)
    got = g.host(g.ops.QLinearMatMul(g.dev(a), 0.02, 117, bd, 0.005, 4, s_y, 128, g.dev(bias)))
    np.testing.assert_array_equal(got[rows], oracle.qlinear_matmul_int(a[rows], 0.02, 117, b, 0.005, 4, s_y, 128, bias=bias))
