"""bf16 / f16 products whose sizes are no multiples of a tile: the
direct-to-LDS kernel with bounds (rows a multiple of 8), and unaligned rows,
against float64 on the rounded operands."""
import numpy as np
import pytest

import rgpu_amd.gpu as G

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    return G.Gpu(0)


def rounded(a, dt):
    return G.bf16_bits_to_f32(G.f32_to_bf16_bits(a)) if dt == G.BF16 else a.astype(np.float16).astype(np.float32)


# K, M and N around the 64-k stage and the 64, 128 and 256 tiles; the last
# three have odd rows (the register-staged kernel).
SHAPES = [(8, 8, 8), (65, 72, 56), (66, 64, 72), (129, 136, 200), (1000, 1032, 64), (1500, 2040, 136), (264, 2000, 328),
          (4100, 4104, 72), (4100, 1000, 520), (4096, 2048, 192), (4000, 2000, 200), (4096, 2040, 64), (63, 65, 67), (130, 1001, 77), (300, 255, 1003)]


@pytest.mark.parametrize("layout", [G.NN, G.TN, G.NT])
@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("dt", [G.BF16, G.F16])
def test_product_bias_mask_and_colsum(gpu, layout, m, n, k, dt):
    rng = np.random.default_rng(m + 3 * n + 7 * k)
    a, b = (rounded(rng.standard_normal(s).astype(np.float32), dt) for s in ((m, k), (k, n)))
    da = np.ascontiguousarray(a.T if layout == G.TN else a)
    db = np.ascontiguousarray(b.T if layout == G.NT else b)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    exact, mag = a64 @ b64, np.abs(a64) @ np.abs(b64)
    # the products are exact; one rounding of the running sum per MFMA
    tol = ((k + 31) // 32 + 4) * 2.0 ** -23 * mag
    A, B, c = gpu.upload(da, dt), gpu.upload(db, dt), gpu.empty((m, n))
    cs = gpu.empty((1, n)) if layout == G.TN else None
    gpu.gemm(layout, A, B, c, colsum=cs)
    assert np.all(np.abs(gpu.download(c) - exact) <= tol)
    if cs is not None:
        assert np.all(np.abs(gpu.download(cs)[0] - b64.sum(0)) <= k * 2.0 ** -24 * np.abs(b64).sum(0) + 1e-30)
    bias = rng.standard_normal((1, n)).astype(np.float32)
    gpu.gemm(layout, A, B, c, G.EPI_BIAS_RELU, gpu.upload(bias))
    assert np.all(np.abs(gpu.download(c) - np.maximum(exact + bias, 0)) <= tol + 2.0 ** -23 * np.abs(bias))
    if dt == G.BF16:  # bf16 results, masked
        h = gpu.empty((m, n), G.BF16)
        mask = rounded(rng.standard_normal((m, n)).astype(np.float32), dt)
        gpu.gemm(layout, A, B, h, G.EPI_RELU_MASK, gpu.upload(mask, G.BF16))
        got = gpu.download_f32(h)
        assert np.all(np.abs(got - exact * (mask > 0)) <= tol + 2.0 ** -8 * np.abs(exact))


@pytest.mark.parametrize("m,n,k,dt,layout", [
    *((4000, 4000, 200, G.BF16, layout) for layout in (G.NN, G.TN, G.NT)),  # 256 blocks with bounds
    *((4001, 4001, 67, G.BF16, layout) for layout in (G.NN, G.TN, G.NT)),   # register-staged (odd rows)
    (5112, 4096, 520, G.F16, G.NN), (5632, 4088, 512, G.F16, G.NT),         # 320 and 352 blocks: 128x128 tiles
    (5632, 4088, 520, G.F16, G.NT)])                                        # 352 blocks over a longer K: 256x256
def test_large_tiles(gpu, m, n, k, dt, layout):
    """The 256x256 tiles and the rule for a last round of few of them."""
    test_product_bias_mask_and_colsum(gpu, layout, m, n, k, dt)


@pytest.mark.parametrize("m,n,k", [(200, 72, 1024), (200, 72, 1032), (1000, 264, 1096)])
@pytest.mark.parametrize("slices", [1, 3])
def test_column_sums_on_both_sides_of_the_sharing_rule(gpu, m, n, k, slices):
    """Up to 1024 rows a slice the first M tile adds them, beyond it the M tiles
    share them: the same sums, to the rounding of their order."""
    rng = np.random.default_rng(k)
    a, b = (rounded(rng.standard_normal(s).astype(np.float32), G.BF16) for s in ((k * slices, m), (k * slices, n)))
    c, cs = gpu.empty((m, n)), gpu.empty((1, n))
    A, B = gpu.upload(a, G.BF16), gpu.upload(b, G.BF16)
    if slices == 1:
        gpu.matmul_at_b(A, B, c, colsum=cs)
    else:
        gpu.split_k(A, B, c, gpu.empty((slices * (m * n + n),)), slices, True, colsum=cs)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    kk = k * slices
    assert np.all(np.abs(gpu.download(cs)[0] - b64.sum(0)) <= kk * 2.0 ** -24 * np.abs(b64).sum(0))
    assert np.all(np.abs(gpu.download(c) - a64.T @ b64) <= ((kk + 31) // 32 + 4) * 2.0 ** -23 * (np.abs(a64).T @ np.abs(b64)))


@pytest.mark.parametrize("layout", [G.NN, G.TN, G.NT])
def test_what_lies_past_an_edge_does_not_reach_the_result(gpu, layout):
    """A row of infinities next to another row's K remainder, and operands
    that end where their buffer ends."""
    m, n, k = 136, 72, 72
    rng = np.random.default_rng(3)
    a, b = (rounded(rng.standard_normal(s).astype(np.float32), G.BF16) for s in ((m, k), (k, n)))
    a[50, :] = np.inf
    b[:, 20] = np.inf
    da = np.ascontiguousarray(a.T if layout == G.TN else a)
    db = np.ascontiguousarray(b.T if layout == G.NT else b)
    c = gpu.empty((m, n))
    gpu.gemm(layout, gpu.upload(da, G.BF16), gpu.upload(db, G.BF16), c)
    got = gpu.download(c)
    keep = np.ix_([i for i in range(m) if i != 50], [j for j in range(n) if j != 20])
    a0, b0 = a.copy(), b.copy()
    a0[50], b0[:, 20] = 0, 0
    exact, mag = a0.astype(np.float64) @ b0, np.abs(a0).astype(np.float64) @ np.abs(b0)
    assert np.all(np.abs(got - exact)[keep] <= 8 * 2.0 ** -23 * mag[keep])
    assert not np.isfinite(got[50]).any() and not np.isfinite(got[:, 20]).any()


@pytest.mark.parametrize("dt", [G.BF16, G.F16])
@pytest.mark.parametrize("m,n,k,slices", [(72, 136, 1000, 4), (520, 264, 5000, 16), (72, 72, 200, 8), (130, 77, 3001, 8)])
def test_slices(gpu, dt, m, n, k, slices):
    """K slices of a ragged product: the last slice cut, or empty."""
    rng = np.random.default_rng(k)
    a, b = (rounded(rng.standard_normal(s).astype(np.float32), dt) for s in ((k, m), (k, n)))
    dw, cs = gpu.empty((m, n)), gpu.empty((1, n))
    gpu.split_k(gpu.upload(a, dt), gpu.upload(b, dt), dw, gpu.empty((slices * (m * n + n),)), slices, True, colsum=cs)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    tol = ((k + 31) // 32 + slices + 4) * 2.0 ** -23 * (np.abs(a64).T @ np.abs(b64))
    assert np.all(np.abs(gpu.download(dw) - a64.T @ b64) <= tol)
    assert np.all(np.abs(gpu.download(cs)[0] - b64.sum(0)) <= k * 2.0 ** -24 * np.abs(b64).sum(0))


@pytest.mark.parametrize("dims", [[128, 256, 128], [72, 200, 101]])
@pytest.mark.parametrize("bad", [False, True])
def test_reduction_of_a_split_gradient_flags_what_is_not_finite(gpu, dims, bad):
    """Batch 1024: every dW of the plan is summed over K slices, and that
    reduction alone sets the overflow flag (four columns at a time, or one)."""
    batch = 1024
    rng = np.random.default_rng(7)
    params = []
    for i, o in zip(dims, dims[1:]):
        params += [rng.standard_normal((i, o)).astype(np.float32) / 16, np.zeros((1, o), np.float32)]
    x = rng.standard_normal((batch, dims[0])).astype(np.float32)
    if bad:
        x[1000, 5] = np.inf  # one row of the last slice (3e38 times weights of 1/16 would stay finite)
    y = G.upload_labels(gpu, rng.integers(0, dims[-1], batch).astype(np.uint32))
    mlp = G.GpuMlp.from_params(gpu, params, batch, 1e-3, precision="bf16", loss_scale=1024.0)
    w0 = mlp.weights()
    mlp.step(gpu.upload(x, G.BF16), y)
    assert mlp.overflow() == bad
    same = all(np.array_equal(a, b) for a, b in zip(w0, mlp.weights()))
    assert same == bad
