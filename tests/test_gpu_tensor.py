"""rakkan_tensor_v1 matmul / matmul_t, quantize and scale on the GPU against
the oracle, bit for bit (internal/sandbox/tensor.go:286-339, 366-387,
445-461; the reference's cases in internal/sandbox/tensor_test.go)."""
import numpy as np
import pytest

import rkhip
from oracle import oracle
from test_gpu_matvec import awkward

pytestmark = pytest.mark.gpu


def bits(x):
    return np.ascontiguousarray(x).view(np.uint32)


@pytest.mark.parametrize("m,k,n", [(7, 33, 5), (64, 64, 64), (100, 257, 70), (1, 4096, 1), (130, 1000, 33),
                                   (33, 3, 129)])
def test_f32_matmul_and_matmul_t(dev, m, k, n):
    rng = np.random.default_rng(m * 1000 + k + n)
    a = awkward(rng, m * k, 1.0).reshape(m, k)
    b = awkward(rng, k * n, 1.0).reshape(k, n)
    want = oracle.tensor_matmul_f32(a, b, False)
    assert np.array_equal(bits(dev.tensor_matmul(a, b)), bits(want))
    bt = np.ascontiguousarray(b.T)
    assert np.array_equal(bits(dev.tensor_matmul(a, bt, transposed=True)), bits(want))


def test_f32_inf_times_zero_is_canonical(dev):
    """TestTensorNaNIsCanonical: Inf·0 -> 0x7fc00000; and a NaN input with
    another payload comes out canonical too."""
    c = dev.tensor_matmul(np.array([[np.inf]], np.float32), np.array([[0]], np.float32))
    assert int(bits(c)[0, 0]) == 0x7FC00000
    odd = np.array([0x7FA00001], np.uint32).view(np.float32)
    c = dev.tensor_matmul(np.array([[1.0, odd[0]]], np.float32), np.array([[1.0], [1.0]], np.float32))
    assert int(bits(c)[0, 0]) == 0x7FC00000


def test_i8_closed_form(dev):
    """TestInt8MatmulIsExact (tensor_test.go:69-95)."""
    a = (np.arange(3 * 64) % 255 - 127).astype(np.int8).reshape(3, 64)
    b = (127 - np.arange(64 * 2) % 200).astype(np.int8).reshape(64, 2)
    c = dev.tensor_matmul(a, b)
    assert c.dtype == np.int32
    assert np.array_equal(c, oracle.tensor_matmul_i8(a, b, False))


@pytest.mark.parametrize("m,k,n", [(64, 256, 64), (70, 1000, 130), (1, 31, 1), (200, 3000, 17), (5, 70000, 9)])
def test_i8_matmul_and_matmul_t(dev, m, k, n):
    rng = np.random.default_rng(m + k * 3 + n * 7)
    a = rng.integers(-128, 128, (m, k), dtype=np.int16).astype(np.int8)
    b = rng.integers(-128, 128, (k, n), dtype=np.int16).astype(np.int8)
    want = oracle.tensor_matmul_i8(a, b, False)
    assert np.array_equal(dev.tensor_matmul(a, b), want)
    assert np.array_equal(dev.tensor_matmul(a, np.ascontiguousarray(b.T), transposed=True), want)


def test_i8_wraps_like_go_int32(dev):
    k = 140000
    a = np.full((2, k), 127, np.int8)
    b = np.full((k, 3), 127, np.int8)
    b[:, 1] = -128
    b[::7, 2] = -128
    assert np.array_equal(dev.tensor_matmul(a, b), oracle.tensor_matmul_i8(a, b, False))


def test_quantize(dev):
    a = np.array([0.25, 0.75, -0.25, 1000, -1000], np.float32)
    assert list(dev.tensor_quantize(a, 0.5)) == [0, 2, 0, 127, -127]
    rng = np.random.default_rng(3)
    x = awkward(rng, 200000, 60.0)
    x[:10] = [2.5, -2.5, 3.5, 126.5, 127.5, -127.5, np.inf, -np.inf, np.nan, -0.0]
    for k in (0.5, 0.37, 3.0, 1e-30):
        assert np.array_equal(dev.tensor_quantize(x, k), oracle.tensor_quantize(x, k)), k


def test_scale(dev):
    assert list(dev.tensor_scale(np.array([4, -6], np.int32), 0.5)) == [2.0, -3.0]
    rng = np.random.default_rng(4)
    i = rng.integers(-(1 << 31), 1 << 31, 100000, dtype=np.int64).astype(np.int32)
    assert np.array_equal(bits(dev.tensor_scale(i, 0.37)), bits(oracle.tensor_scale_i32(i, 0.37)))
    f = awkward(rng, 100000, 1e30)
    f[:3] = [np.inf, np.nan, -np.inf]
    want = (f * np.float32(0.0)).astype(np.float32)
    want[np.isnan(want)] = np.array([0x7FC00000], np.uint32).view(np.float32)[0]
    assert np.array_equal(bits(dev.tensor_scale(f, 0.0)), bits(want))


def test_argument_errors(dev):
    f = np.ones((2, 2), np.float32)
    with pytest.raises(rkhip.RKError) as e:
        dev.tensor_matmul(f, np.ones((3, 2), np.float32))
    assert e.value.code == -1
    L = rkhip.lib()
    c = np.empty(4, np.int32)
    i32 = np.ones(4, np.int32)
    # i32 inputs are rejected as by tenMatmul (tenErrArgs)
    assert L.rk_tensor_matmul(dev.h, rkhip.TENSOR_I32, 0, 2, 2, 2, rkhip._ptr(i32), rkhip._ptr(i32),
                              rkhip._ptr(c)) == -1
    with pytest.raises(rkhip.RKError):
        dev.tensor_quantize(f, 0.0)
    with pytest.raises(rkhip.RKError):
        dev.tensor_scale(np.ones(3, np.int8), 1.0)


# Sizes about the tiles' edges (32 outputs a side in f32; 128, 64 and 32 in
# i8, by the number of tiles), the staged slices' (64 positions; 128, 256 and
# 512) and the loads' (4 floats, 16 bytes); int8 on device pointers off their
# alignment too.
TILE_SHAPES = [(32, 64, 32), (33, 65, 31), (31, 63, 97), (1, 1, 1), (2, 15, 3), (64, 128, 260), (513, 17, 65),
               (300, 130, 70)]


@pytest.mark.parametrize("m,k,n", TILE_SHAPES + [(1024, 48, 1030)])
def test_f32_tiles(dev, m, k, n):
    rng = np.random.default_rng(m + 31 * k + 7 * n)
    a = awkward(rng, m * k, 1.0).reshape(m, k)
    b = awkward(rng, k * n, 1.0).reshape(k, n)
    want = bits(oracle.tensor_matmul_f32(a, b, False))
    assert np.array_equal(bits(dev.tensor_matmul(a, b)), want)
    assert np.array_equal(bits(dev.tensor_matmul(a, np.ascontiguousarray(b.T), transposed=True)), want)


@pytest.mark.parametrize("m,k,n", TILE_SHAPES + [(70, 511, 33), (70, 513, 31), (1000, 257, 700), (1025, 16, 1021),
                                                 (2048, 129, 1600), (1793, 143, 1795)])
@pytest.mark.parametrize("off", [0, 1, 6])
def test_i8_tiles(dev, m, k, n, off):
    rng = np.random.default_rng(m + 31 * k + 7 * n)
    a = rng.integers(-128, 128, (m, k), dtype=np.int16).astype(np.int8)
    b = rng.integers(-128, 128, (k, n), dtype=np.int16).astype(np.int8)
    want = oracle.tensor_matmul_i8(a, b, False)

    def words(v):  # the bytes, `off` bytes into their words
        v = np.concatenate((np.zeros(off, np.int8), v.ravel()))
        return np.concatenate((v, np.zeros(-v.size % 4, np.int8))).view(np.float32)

    at_a, at_b, at_c = 0, words(a).size, words(a).size + words(b).size
    arena = dev.arena(at_c + m * n, at_c + m * n)
    for transposed, y in ((0, b), (1, np.ascontiguousarray(b.T))):
        q = arena.begin()
        q.write(at_a, words(a))
        q.write(at_b, words(y))
        q.write(at_c, np.full(m * n, -1, np.int32).view(np.float32))
        q.submit()
        dev._check(rkhip.lib().rk_tensor_matmul_device(dev.h, rkhip.TENSOR_I8, transposed, m, k, n,
                                                       arena.device_ptr(at_a) + off, arena.device_ptr(at_b) + off,
                                                       arena.device_ptr(at_c), None))
        q = arena.begin()
        got = q.read(at_c, m * n)
        q.submit()
        assert np.array_equal(got.view(np.int32).reshape(m, n), want)
    arena.free()


# More tiles than one grid dimension takes (2^24 workgroups of 256 threads).
def test_f32_more_tiles_than_a_grid_dimension(dev):
    m = n = 1 << 17
    rng = np.random.default_rng(17)
    a, b = rng.normal(0, 1, (2, m)).astype(np.float32)
    at_c = 2 * m
    arena = dev.arena(at_c + m * n, 2 * m + 8 * n)
    try:
        q = arena.begin()
        q.write(0, a)
        q.write(m, b)
        q.submit()
        dev._check(rkhip.lib().rk_tensor_matmul_device(dev.h, rkhip.TENSOR_F32, 0, m, 1, n, arena.device_ptr(0),
                                                       arena.device_ptr(m), arena.device_ptr(at_c), None))
        rows = [0, 1, 31, 32, 65537, 100003, m - 33, m - 1]
        q = arena.begin()
        got = [q.read(at_c + i * n, n) for i in rows]
        q.submit()
        for i, g in zip(rows, got):
            assert np.array_equal(bits(np.asarray(g)), bits(np.float32(0) + a[i] * b)), i
    finally:
        arena.free()


@pytest.mark.parametrize("m,k,n", [(33, 65, 31), (64, 128, 260), (2, 15, 3), (40, 200, 70)])
@pytest.mark.parametrize("off", [0, 1])
def test_f32_infinities_and_nans(dev, m, k, n, off):
    """The matrix core's products of infinities, NaNs of any payload and
    zeros of both signs, and their sums, on device pointers at and off their
    16-byte alignment."""
    rng = np.random.default_rng(m + 31 * k + 7 * n)
    odd = np.array([0x7F800000, 0xFF800000, 0x7FA00001, 0xFFC12345, 0x80000000, 0, 0x7F7FFFFF, 1], np.uint32).view(np.float32)

    def draw(rows, cols):
        v = awkward(rng, rows * cols, 1.0)
        hit = rng.random(v.size) < 2.0 / k  # most rows and columns hold one or two
        v[hit] = rng.choice(odd, hit.sum())
        return v.reshape(rows, cols)

    a, b = draw(m, k), draw(k, n)
    want = bits(oracle.tensor_matmul_f32(a, b, False))
    at_a, at_b = off, (m * k + 3 & ~3) + off
    at_c = at_b + k * n
    arena = dev.arena(at_c + m * n, at_c + 2 * m * n)
    try:
        for transposed, y in ((0, b), (1, np.ascontiguousarray(b.T))):
            q = arena.begin()
            q.write(at_a, a.ravel())
            q.write(at_b, y.ravel())
            q.submit()
            dev._check(rkhip.lib().rk_tensor_matmul_device(dev.h, rkhip.TENSOR_F32, transposed, m, k, n,
                                                           arena.device_ptr(at_a), arena.device_ptr(at_b),
                                                           arena.device_ptr(at_c), None))
            q = arena.begin()
            got = q.read(at_c, m * n)
            q.submit()
            assert np.array_equal(bits(np.asarray(got)).reshape(m, n), want)
    finally:
        arena.free()


# More than 65536 positions (the matrix core's sums start again and are added
# with wraparound) in the 64 x 64 and the 128 x 64 tiles. a_ip = u_i s_p and
# b_pj = v_j t_p, so c_ij = u_i v_j sum(s_p t_p).
@pytest.mark.parametrize("m,n", [(768, 704), (2048, 1024)])
def test_i8_restarts_in_the_wide_tiles(dev, m, n):
    rng = np.random.default_rng(m)
    k = 131072 + 100
    u, v = rng.integers(-127, 128, m), rng.integers(-127, 128, n)
    s = np.ones(k, np.int8)
    t = np.ones(k, np.int8)
    t[rng.integers(0, k, 1000)] = -1  # 127 * 127 * 129000 leaves int32's range
    u[:3], v[:2] = 127, (127, -127)
    want = (np.outer(u, v).astype(np.int64) * int(t.astype(np.int64).sum())).astype(np.uint32).view(np.int32)
    a = u.astype(np.int8)[:, None] * s
    b = t[:, None] * v.astype(np.int8)
    assert np.array_equal(dev.tensor_matmul(a, b), want)
    assert np.array_equal(dev.tensor_matmul(a, np.ascontiguousarray(b.T), transposed=True), want)
