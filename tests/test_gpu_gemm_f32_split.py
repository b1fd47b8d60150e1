"""f32 products on the bf16 matrix units (gemm_f32.hip, F32Split): tile edges,
K remainders, unaligned rows, epilogues, and operands that are not finite,
against float64."""
import numpy as np
import pytest

import rgpu_amd.gpu as G

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    return G.Gpu(0)


def bound(k, mag):
    """|error| of an element whose |A|·|B| is mag: one rounding of the running
    sum per MFMA (32 k) in the main accumulator and as many, 2^-8 smaller, in
    the other; the parts left out (2^-26); the epilogue's.  The matrix unit may
    truncate, hence 2^-23."""
    return ((k + 31) // 32 + 4) * 2.0 ** -23 * mag + 1e-37


def operands(layout, m, n, k, rng):
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    dev_a = a.T if layout == G.TN else a
    dev_b = b.T if layout == G.NT else b
    return a, b, np.ascontiguousarray(dev_a), np.ascontiguousarray(dev_b)


# Around the edges of the 64x32, 64x64 and 128x64 tiles, rows that start off
# 16 bytes, and K at the edges of the 64-k stage and of the rules on K.
SHAPES = [(65, 33, 1), (65, 31, 63), (66, 34, 64), (67, 65, 65), (129, 127, 129), (130, 64, 191), (128, 192, 512),
          (128, 192, 544), (1030, 1033, 130), (2050, 1090, 70), (127, 30, 1000), (70, 2500, 333), (1, 40, 700)]


@pytest.mark.parametrize("layout", [G.NN, G.TN, G.NT])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_product_against_float64(gpu, layout, m, n, k):
    rng = np.random.default_rng(m * 31 + n * 7 + k)
    a, b, da, db = operands(layout, m, n, k, rng)
    c = gpu.empty((m, n))
    cs = gpu.empty((1, n)) if layout == G.TN else None
    gpu.gemm(layout, gpu.upload(da), gpu.upload(db), c, colsum=cs)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    assert np.all(np.abs(gpu.download(c) - a64 @ b64) <= bound(k, np.abs(a64) @ np.abs(b64)))
    if cs is not None:
        assert np.all(np.abs(gpu.download(cs)[0] - b64.sum(0)) <= (k / 2 + 8) * 2.0 ** -24 * np.abs(b64).sum(0))


@pytest.mark.parametrize("layout", [G.NN, G.TN, G.NT])
@pytest.mark.parametrize("m,n,k", [(257, 133, 1), (257, 33, 2), (640, 2033, 2), (640, 2033, 96), (640, 2033, 97),
                                   (1856, 1200, 128), (1856, 1200, 129), (1856, 1200, 192), (1856, 1200, 193)])
def test_short_products_against_float64(gpu, layout, m, n, k):
    """Both sides of the rule on K.  A product of one k is the rounded product,
    one of two the rounded sum of a rounded and an exact one, whatever the tile."""
    rng = np.random.default_rng(m + n + k)
    a, b, da, db = operands(layout, m, n, k, rng)
    c = gpu.empty((m, n))
    gpu.gemm(layout, gpu.upload(da), gpu.upload(db), c)
    got, a64, b64 = gpu.download(c), a.astype(np.float64), b.astype(np.float64)
    mag = np.abs(a64) @ np.abs(b64)
    if k == 1:
        assert np.array_equal(got, a * b)
    assert np.all(np.abs(got - a64 @ b64) <= (2.0 * 2.0 ** -24 * mag if k == 2 else bound(k, mag)))


@pytest.mark.parametrize("rows,din,dout", [(3000, 900, 40), (2100, 2000, 100), (2100, 2000, 200), (600, 70, 2)])
def test_pair_of_a_short_product_gives_the_bits_of_its_products(gpu, rows, din, dout):
    rng = np.random.default_rng(rows)
    x, d, w = (gpu.upload(rng.standard_normal(s).astype(np.float32)) for s in ((rows, din), (rows, dout), (din, dout)))
    dx, dw, db = gpu.empty((rows, din)), gpu.empty((din, dout)), gpu.empty((1, dout))
    gpu.linear_backward(x, d, w, dx, dw, db)
    dx1, dw1, db1 = gpu.empty((rows, din)), gpu.empty((din, dout)), gpu.empty((1, dout))
    gpu.matmul_at_b(x, d, dw1, colsum=db1)
    gpu.matmul_a_bt(d, w, dx1)
    for got, want in ((dx, dx1), (dw, dw1), (db, db1)):
        assert gpu.download(got).tobytes() == gpu.download(want).tobytes()


@pytest.mark.parametrize("m,n,k", [(129, 65, 200), (256, 128, 576), (300, 77, 1000)])
def test_epilogues(gpu, m, n, k):
    rng = np.random.default_rng(m + n + k)
    a, b, da, db = operands(G.NN, m, n, k, rng)
    bias = rng.standard_normal((1, n)).astype(np.float32)
    mask = rng.standard_normal((m, n)).astype(np.float32)
    exact = a.astype(np.float64) @ b.astype(np.float64)
    tol = bound(k, np.abs(a).astype(np.float64) @ np.abs(b) + np.abs(bias))
    c = gpu.empty((m, n))
    gpu.gemm(G.NN, gpu.upload(da), gpu.upload(db), c, G.EPI_BIAS, gpu.upload(bias))
    assert np.all(np.abs(gpu.download(c) - (exact + bias)) <= tol)
    gpu.gemm(G.NN, gpu.upload(da), gpu.upload(db), c, G.EPI_BIAS_RELU, gpu.upload(bias))
    assert np.all(np.abs(gpu.download(c) - np.maximum(exact + bias, 0)) <= tol)
    gpu.gemm(G.NT, gpu.upload(da), gpu.upload(np.ascontiguousarray(b.T)), c, G.EPI_RELU_MASK, gpu.upload(mask))
    assert np.all(np.abs(gpu.download(c) - exact * (mask > 0)) <= tol)


@pytest.mark.parametrize("layout", [G.NN, G.TN, G.NT])
@pytest.mark.parametrize("slices", [1, 3, 5])
def test_slices_and_pair(gpu, layout, slices):
    """K slices that end inside a stage (and an empty last one) against the
    float64 product; the paired backward gives the bits of its two products."""
    m, n, k = 100, 70, 288
    rng = np.random.default_rng(slices)
    a, b, da, db = operands(layout, m, n, k, rng)
    c = gpu.empty((m, n))
    if layout != G.NT:
        gpu.split_k(gpu.upload(da), gpu.upload(db), c, gpu.empty((slices * m * n,)), slices, layout == G.TN)
        a64, b64 = a.astype(np.float64), b.astype(np.float64)
        assert np.all(np.abs(gpu.download(c) - a64 @ b64) <= 2 * bound(k, np.abs(a64) @ np.abs(b64)))
        return
    x, d, w = (gpu.upload(rng.standard_normal(s).astype(np.float32)) for s in ((300, 90), (300, 70), (90, 70)))
    dx, dw, dbv = gpu.empty((300, 90)), gpu.empty((90, 70)), gpu.empty((1, 70))
    gpu.linear_backward(x, d, w, dx, dw, dbv)
    dx1, dw1, db1 = gpu.empty((300, 90)), gpu.empty((90, 70)), gpu.empty((1, 70))
    gpu.matmul_at_b(x, d, dw1, colsum=db1)
    gpu.matmul_a_bt(d, w, dx1)
    for got, want in ((dx, dx1), (dw, dw1), (dbv, db1)):
        assert gpu.download(got).tobytes() == gpu.download(want).tobytes()


@pytest.mark.parametrize("layout", [G.NN, G.TN, G.NT])
def test_operands_that_are_not_finite(gpu, layout):
    """Infinities, NaN, sums that overflow and values next to the largest give
    what f32 arithmetic gives; other rows and columns keep their values."""
    m, n, k = 200, 96, 150
    rng = np.random.default_rng(5)
    a, b, _, _ = operands(layout, m, n, k, rng)
    a[0, 3], a[20, 7], a[40, 149] = np.inf, np.nan, -np.inf
    b[7, 10], b[100, 50] = np.inf, np.nan
    b[3, 5], b[3, 6] = 0.0, -1.0  # inf * 0 is NaN, inf * -1 is -inf
    a[60, :], a[60, 0] = 0.0, np.float32(3.4e38)  # rounds to infinity in bf16
    b[0, :] = 0.5
    a[80, :] = np.float32(3e38)
    b[:, 20] = 1.0  # row 80, column 20 overflows
    with np.errstate(all="ignore"):
        want = (a.astype(np.float64) @ b.astype(np.float64))
        want = np.where(np.abs(want) > 3.4028235e38, np.sign(want) * np.inf, want)
    da = np.ascontiguousarray(a.T if layout == G.TN else a)
    db = np.ascontiguousarray(b.T if layout == G.NT else b)
    c = gpu.empty((m, n))
    gpu.gemm(layout, gpu.upload(da), gpu.upload(db), c)
    got = gpu.download(c)
    rows = [i for i in range(m) if i != 80]  # row 80 may overflow on the way, in an order of its own
    assert np.array_equal(np.isnan(got[rows]), np.isnan(want[rows]))
    assert np.array_equal(np.isposinf(got[rows]), np.isposinf(want[rows]))
    assert np.array_equal(np.isneginf(got[rows]), np.isneginf(want[rows]))
    assert got[80, 20] == np.inf
    fin = np.isfinite(want) & np.isfinite(got)
    with np.errstate(all="ignore"):
        mag = np.abs(np.where(np.isfinite(a), a, 0)).astype(np.float64) @ np.abs(np.where(np.isfinite(b), b, 0))
    fin[80] = False
    assert np.all(np.abs(np.where(fin, got, 0) - np.where(fin, want, 0)) <= bound(k, mag))


@pytest.mark.parametrize("layout", [G.NN, G.TN, G.NT])
@pytest.mark.parametrize("scale", [0, 50])
@pytest.mark.parametrize("m,n,k", [(129, 65, 200), (300, 31, 333)])
def test_infinities_among_finite_operands(gpu, layout, scale, m, n, k):
    """A tile that holds infinities and NaN takes them from the leading
    products where its sums cannot overflow (scale 0), and is computed again
    where they can (2^50: products of 2^100); whole rows of NaN."""
    rng = np.random.default_rng(m + scale)
    a, b, _, _ = operands(layout, m, n, k, rng)
    a, b = np.ldexp(a, scale).astype(np.float32), np.ldexp(b, scale).astype(np.float32)
    a[3, k - 1], a[17, 5], a[17, 6], a[100, :] = -np.inf, np.inf, np.inf, np.nan
    b[5, 7], b[6, 7], b[5, 9], b[k - 1, 30] = 1.0, -1.0, 0.0, np.inf  # row 17: inf - inf, inf * 0
    with np.errstate(all="ignore"):
        want = a.astype(np.float64) @ b.astype(np.float64)
        mag = np.abs(np.where(np.isfinite(a), a, 0)).astype(np.float64) @ np.abs(np.where(np.isfinite(b), b, 0))
    c = gpu.empty((m, n))
    gpu.gemm(layout, gpu.upload(np.ascontiguousarray(a.T if layout == G.TN else a)),
             gpu.upload(np.ascontiguousarray(b.T if layout == G.NT else b)), c)
    got = gpu.download(c)
    fin = np.isfinite(want)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)].astype(np.float32))
    assert np.all(np.abs(got[fin] - want[fin]) <= bound(k, mag)[fin])


def test_small_magnitudes_keep_their_precision(gpu):
    """Operands around 2^-90: the parts of the split stay above the smallest
    subnormal bf16, so the relative error is that of ordinary values."""
    m, n, k = 128, 128, 640
    rng = np.random.default_rng(9)
    a, b, _, _ = operands(G.NN, m, n, k, rng)
    s = np.float32(2.0 ** -90)
    c = gpu.empty((m, n))
    gpu.gemm(G.NN, gpu.upload(a * s), gpu.upload(b), c)
    mag = np.abs(a).astype(np.float64) @ np.abs(b)
    assert np.all(np.abs(gpu.download(c) / np.float64(s) - a.astype(np.float64) @ b) <= bound(k, mag))


@pytest.mark.parametrize("layout", [G.NN, G.TN, G.NT])
@pytest.mark.parametrize("ea,eb", [(-108, 100), (-115, 100), (-128, 100), (-140, 100), (100, -128), (-126, 60),
                                   (112, -100), (100, 20), (60, 60)])
def test_magnitudes_at_the_ends_of_the_range(gpu, layout, ea, eb):
    """Operands whose last bits lie below the smallest bf16, f32 subnormals
    among them, against large ones, so that the results are ordinary numbers;
    and operands and sums near the largest f32: the error stays that of a
    product of ordinary values (an operand's own bits are exact)."""
    m, n, k = 129, 65, 200
    rng = np.random.default_rng(ea + 1000)
    a, b, _, _ = operands(layout, m, n, k, rng)
    a, b = np.ldexp(a, ea).astype(np.float32), np.ldexp(b, eb).astype(np.float32)
    c = gpu.empty((m, n))
    gpu.gemm(layout, gpu.upload(np.ascontiguousarray(a.T if layout == G.TN else a)),
             gpu.upload(np.ascontiguousarray(b.T if layout == G.NT else b)), c)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    assert np.all(np.abs(gpu.download(c) - a64 @ b64) <= bound(k, np.abs(a64) @ np.abs(b64)))


@pytest.mark.parametrize("m,n,k", [(512, 10, 256), (100, 32, 200), (65, 17, 129), (64, 33, 128)])
def test_bias_gradient_of_a_narrow_layer_is_added_in_row_order(gpu, m, n, k):
    rng = np.random.default_rng(m + n + k)
    a, b, da, db = operands(G.TN, m, n, k, rng)
    c, cs = gpu.empty((m, n)), gpu.empty((1, n))
    gpu.matmul_at_b(gpu.upload(da), gpu.upload(db), c, colsum=cs)
    mag = np.abs(a).astype(np.float64) @ np.abs(b)
    assert np.all(np.abs(gpu.download(c) - a.astype(np.float64) @ b) <= bound(k, mag))
    want = np.add.accumulate(b, axis=0, dtype=np.float32)[-1]  # one by one, left to right: the same bits
    assert np.array_equal(gpu.download(cs)[0], want)


@pytest.mark.parametrize("layout", [G.NN, G.TN, G.NT])
def test_more_rows_than_one_grid_holds(gpu, layout):
    """2^30 rows of one column, the most the entry point takes, need 2^24 blocks
    of 256 threads: every row is computed.  Sums of ones are exact."""
    m = 2 ** 30
    a, c, total = gpu.zeros((1, m) if layout == G.TN else (m, 1)), gpu.zeros((m, 1)), gpu.empty((1,))
    gpu.map("offset", a, a, 1.0)
    cs = gpu.empty((1, 1)) if layout == G.TN else None
    gpu.gemm(layout, a, gpu.upload(np.full((1, 1), 2, np.float32)), c, colsum=cs)
    gpu.sum_all(c, total, m)
    assert gpu.download(total)[0] == 2
    if cs is not None:
        assert gpu.download(cs)[0, 0] == 2
