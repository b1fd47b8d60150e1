"""Row kernels of the tape (softmax, its VJP, softmax cross-entropy from the
logits) at the row lengths and counts where their lane groups change."""
import numpy as np
import pytest

import rgpu_amd.gpu as G

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    return G.Gpu(0)


# Row lengths at the edges of every lane group (4, 8, .., 64 lanes; a wave with
# 4 or 16 registers; rows through LDS in chunks).
COLS = [1, 4, 5, 8, 9, 16, 17, 32, 33, 64, 65, 256, 257, 1000, 1024, 1025, 4096, 4097, 9001]


def f64_softmax(z):
    e = np.exp(z - z.max(1, keepdims=True))
    return e / e.sum(1, keepdims=True)


# Relative error of p: the sum of `cols` positive terms in order (cols / 2 eps),
# exp and the division (a few ulp), and the rounding of z - max, which exp
# multiplies by |z - max|.
EPS = float(np.finfo(np.float32).eps)


@pytest.mark.parametrize("cols", COLS)
@pytest.mark.parametrize("rows", [1, 67, 4099])
def test_softmax_and_vjp(gpu, rows, cols):
    if rows * cols > 5_000_000:
        pytest.skip("the small row counts cover this row length")
    r = np.random.default_rng(rows * 10007 + cols)
    z = (r.standard_normal((rows, cols)) * 3).astype(np.float32)
    g = r.standard_normal((rows, cols)).astype(np.float32)
    zd, gd, p, dx = gpu.upload(z), gpu.upload(g), gpu.empty((rows, cols)), gpu.empty((rows, cols))
    gpu.softmax_rows(zd, p)
    gpu.softmax_rows_vjp(p, gd, dx)
    z64, g64 = z.astype(np.float64), g.astype(np.float64)
    want = f64_softmax(z64)
    span = (z64.max(1, keepdims=True) - z64 + 8 + cols / 2) * EPS
    got = gpu.download(p)
    assert np.all(np.abs(got - want) <= want * span)
    # the VJP's dot is added in column order, each product and sum rounded on
    # its own (ops.rs:291-309): the same bits
    dot = np.add.accumulate(g * got, axis=1, dtype=np.float32)[:, -1:]
    assert gpu.download(dx).tobytes() == (got * (g - dot)).tobytes()
    # in place: the same bits
    gpu.softmax_rows(zd, zd)
    assert gpu.download(zd).tobytes() == got.tobytes()
    gpu.softmax_rows_vjp(p, gd, gd)
    assert gpu.download(gd).tobytes() == gpu.download(dx).tobytes()


@pytest.mark.parametrize("rows,cols", [(1, 1), (512, 16), (513, 16), (128, 64), (129, 64), (16, 1000), (127, 1000),
                                       (128, 1000), (4, 4097), (40, 4097), (3000, 5), (0, 7)])
def test_xent_from_logits_blocks(gpu, rows, cols):
    """One block, several, and the last one partly filled: P − Y as
    softmax_rows gives it, the value against float64."""
    r = np.random.default_rng(rows + 31 * cols)
    z = (r.standard_normal((rows, cols)) * 3).astype(np.float32)
    y = np.zeros((rows, cols), np.float32)
    y[np.arange(rows), r.integers(0, cols, rows)] = 1.0
    zd, yd, p, d, v = gpu.upload(z), gpu.upload(y), gpu.empty((rows, cols)), gpu.empty((rows, cols)), gpu.empty(())
    gpu.softmax_rows(zd, p)
    gpu.loss(G.LOSS_SOFTMAX_XENT_LOGITS, zd, yd, v, d)
    value = float(gpu.download(v))
    if rows == 0:
        assert np.isnan(value)  # 0 / 0, as the reference's mean over no rows
        return
    assert gpu.download(d).tobytes() == (gpu.download(p) - y).tobytes()
    want = -np.log(np.maximum((f64_softmax(z.astype(np.float64)) * y).sum(1), 1e-12)).mean()
    assert abs(value - want) <= 2e-6 * max(1.0, abs(want))


@pytest.mark.parametrize("cols", [2, 4, 5, 7, 8])
@pytest.mark.parametrize("rows", [1, 255, 256, 257])
def test_xent_from_logits_narrow_rows(gpu, rows, cols):
    """A thread per row up to 7 columns, lane groups from 8 on, and one block
    or several."""
    test_xent_from_logits_blocks(gpu, rows, cols)


def test_rows_that_are_not_finite(gpu):
    """A NaN or +inf makes its own row NaN, a row of -inf too; -inf next to
    finite values is a probability of zero.  Other rows are untouched."""
    z = np.zeros((6, 70), np.float32)
    z[0, 69], z[1, 3], z[2, :], z[3, 5] = np.nan, np.inf, -np.inf, -np.inf
    p = gpu.empty(z.shape)
    gpu.softmax_rows(gpu.upload(z), p)
    got = gpu.download(p)
    assert np.isnan(got[0]).all() and np.isnan(got[2]).all() and np.isnan(got[1, 3])
    assert got[3, 5] == 0.0 and np.isclose(got[3, 0], 1 / 69)
    assert np.allclose(got[4:], 1 / 70)


# Rows at the edges of the column kernel's stages (256) and add batches (32),
# below its range too; columns at the edges of its blocks (16).
@pytest.mark.parametrize("cols", [2, 15, 16, 17, 1000])
@pytest.mark.parametrize("rows", [2, 31, 32, 33, 255, 256, 257, 512, 2083])
def test_reduce_to_columns(gpu, rows, cols):
    x = np.random.default_rng(rows * 10007 + cols).standard_normal((rows, cols)).astype(np.float32)
    x[:, 0] = -0.0  # 0 + -0 stays +0
    x[rows // 2, 1] = np.inf
    out = gpu.empty((1, cols))
    gpu.reduce_to(gpu.upload(x), out)
    # added one by one in row order (tensor.rs:399-438): the same bits
    want = np.add.accumulate(np.concatenate([np.zeros((1, cols), np.float32), x]), axis=0, dtype=np.float32)[-1:]
    assert np.array_equal(gpu.download(out).view(np.uint32), want.view(np.uint32))


def test_more_rows_than_one_grid_holds(gpu):
    """2^26 rows of 33 columns need 2^32 threads, the size of a grid: every row
    of the softmax, its VJP and the loss is computed.

    The sums run over 2.4e9 values, 4096 parts of 256 threads that add 2300
    each one after another, then a tree: off by at most 2400 * 2^-24 = 1.5e-4 of
    their terms' magnitude; the loss's last stage, 256 threads that add 70000
    blocks' parts each, by at most 70300 * 2^-24 = 4.2e-3.  The rows past the
    grid are 6e-2 of them all."""
    rows, cols = 2 ** 26 + 2 ** 22, 33
    p, one, dx = gpu.zeros((rows, cols)), gpu.zeros((rows, cols)), gpu.empty((rows, cols))
    total, value = gpu.empty((1,)), gpu.empty((1,))
    gpu.map("offset", one, one, 1.0)
    gpu.softmax_rows(p, p)  # of zeros: 1/33 everywhere
    gpu.sum_all(p, total, rows)
    assert abs(gpu.download(total)[0] - 1) < 1.5e-4
    gpu.map("offset", one, dx, 1.0)
    gpu.softmax_rows_vjp(p, one, dx)  # p (1 - sum p) = 0
    gpu.map("square", dx, dx)
    gpu.sum_all(dx, total)
    assert gpu.download(total)[0] < 1e-3
    gpu.map("scale", p, one, 0.0)
    gpu.loss(4, one, p, value, dx)  # logits 0, targets 1/33: ln 33, p - y = 0
    assert abs(gpu.download(value)[0] / np.log(33) - 1) < 4.2e-3
    gpu.map("square", dx, dx)
    gpu.sum_all(dx, total)
    assert gpu.download(total)[0] < 1e-3
