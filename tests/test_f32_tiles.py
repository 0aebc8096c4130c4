"""f32 products on tiles of 32 to 256 rows by 128 columns (k_gemm_f32.hip; Backend::matmul, ndarray.rs:549-615) against sums in
64 bits: every height of tile, with the right operand along k (a weight) and along n, columns and rows that end inside a tile,
depths that end inside a step, slices of k of which the last is shorter, batches, a sigmoid on the way out."""
import numpy as np
import pytest

import vectors
from test_f32_operands import assert_f32_sums

lang, nn = vectors.cg.lang, vectors.cg.nn


def product(rank, along_k, act=False):
    def f(b, x, w):
        y = lang.matmul(b, x, lang.transpose(b, rank - 2, rank - 1, w) if along_k else w)
        return [nn.sigmoid(b, y) if act else y]
    return f


# height of the tile in units of 32 rows (test_kernel_choice.py asserts that each size is given it): B, M, N, K
SIZES = [(1, 1, 40, 8196, 516), (1, 3, 70, 2060, 100), (1, 1, 1000, 1000, 1000), (2, 1, 130, 7312, 52), (2, 1, 520, 900, 2060), (2, 32, 300, 300, 64),
         (3, 1, 96, 32000, 132), (3, 1, 700, 2048, 4100), (4, 1, 256, 32000, 60), (5, 1, 155, 32700, 100), (6, 1, 185, 5380, 1404),
         (7, 1, 220, 30000, 100), (8, 1, 8190, 4096, 44), (8, 1, 719, 2820, 1288)]


@pytest.mark.gpu
@pytest.mark.parametrize("along_k", [True, False])
@pytest.mark.parametrize("rows,B,M,N,K", SIZES)
def test_product(hip, rows, B, M, N, K, along_k):
    g = np.random.default_rng(M + K)
    x = g.standard_normal((B, M, K)).astype(np.float32)
    w = g.standard_normal((B, N, K) if along_k else (B, K, N)).astype(np.float32)
    if B == 1:
        x, w = x[0], w[0]
    (got,) = vectors.run(hip, product(x.ndim, along_k), 1, x, w)
    exact = np.matmul(x.astype(np.float64), (np.swapaxes(w, -1, -2) if along_k else w).astype(np.float64))
    assert_f32_sums(exact, got, K, f"{B} x {M} x {N} x {K}")


def with_infinities(x, w):
    """x [.., M, K] and w [.., N, K] with an infinity in row 3, a NaN in the last row and, of several columns, an infinity in the
    last: at the first and the last k, next to what a tile holds past either edge."""
    x, w = x.copy(), w.copy()
    x[..., 3, 0], x[..., -1, -1] = np.inf, np.nan
    if w.shape[-2] > 1:
        w[..., -1, -1] = -np.inf
    return x, w


def assert_infinities(x, w, got):
    """Infinities and NaN where x w^T has them, nowhere else; K f32 additions of rounded products off in the rest."""
    x, w = x.astype(np.float64), np.swapaxes(w, -1, -2).astype(np.float64)
    with np.errstate(invalid="ignore"):
        ref = np.matmul(x, w)
    finite = np.isfinite(ref)
    assert np.array_equal(ref[~finite], got[~finite], equal_nan=True)
    bound = (x.shape[-1] + 1) * 2.0 ** -24 * np.matmul(*(np.abs(np.where(np.isfinite(a), a, 0)) for a in (x, w)))
    assert np.all(np.abs(got[finite] - ref[finite]) <= bound[finite])      # (a NaN is no less than its bound)


# the smallest, on 16 x 16 tiles (test_kernel_choice.py asserts so): rows and columns that end inside one, k that ends inside a chunk of 16
# or a lane's four, gives some wavefronts nothing, or takes more than one group of chunks; a batch
SMALLEST = [(1, 9, 1, 1), (1, 64, 256, 128), (1, 64, 10, 256), (1, 17, 33, 5), (1, 31, 15, 127), (3, 70, 60, 100), (1, 40, 100, 743), (2, 16, 17, 1023),
            (1, 250, 250, 512), (1, 13, 500, 1024)]


@pytest.mark.gpu
@pytest.mark.parametrize("along_k", [True, False])
@pytest.mark.parametrize("B,M,N,K", SMALLEST)
def test_smallest_product(hip, B, M, N, K, along_k):
    test_product(hip, 0, B, M, N, K, along_k)
    if N > 1 and K > 1:
        test_infinities(hip, 0, B, M, N, K, along_k)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(64, 256, 128), (33, 31, 1000)])
def test_smallest_sigmoid(hip, M, N, K):
    test_sigmoid(hip, M, N, K)


@pytest.mark.gpu
@pytest.mark.parametrize("B,M,N,K", [(1, 64, 256, 128), (3, 33, 31, 1000)])
def test_smallest_product_of_columns_and_residual(hip, B, M, N, K):
    """A left operand whose rows lie across memory, and a residual, added by the product's launch."""
    g = np.random.default_rng(K)
    x, w, r = (g.standard_normal(s).astype(np.float32) for s in ((B, K, M), (B, K, N), (B, M, N)))
    hip.launch_counts(reset=True)
    (got,) = vectors.run(hip, lambda b, r, x, w: [r + lang.matmul(b, lang.transpose(b, 1, 2, x), w)], 1, r, x, w)
    counts = hip.launch_counts(reset=True)
    assert sum(counts.values()) == 1, counts
    exact = np.matmul(np.swapaxes(x, 1, 2).astype(np.float64), w.astype(np.float64))
    bound = (K + 1) * 2.0 ** -24 * np.matmul(np.abs(np.swapaxes(x, 1, 2)), np.abs(w)) + 2.0 ** -24 * np.abs(exact + r)
    assert np.all(np.abs(got - (exact + r)) <= bound)


# every height of tile, k in one piece and in slices, a last step of one piece
@pytest.mark.gpu
@pytest.mark.parametrize("along_k", [True, False])
@pytest.mark.parametrize("rows,B,M,N,K", [s for s in SIZES if s[2] * s[3] < 5e6])
def test_infinities(hip, rows, B, M, N, K, along_k):
    g = np.random.default_rng(M + K)
    x, w = with_infinities(*(g.standard_normal(s).astype(np.float32) for s in (((B, M, K), (B, N, K)) if B > 1 else ((M, K), (N, K)))))
    (got,) = vectors.run(hip, product(x.ndim, along_k), 1, x, w if along_k else np.ascontiguousarray(np.swapaxes(w, -1, -2)))
    assert_infinities(x, w, got)


# one launch and slices whose sum applies it; the error of a sigmoid is at most a quarter of its argument's, and its own rounding
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1000, 1000, 1000), (300, 1000, 2060)])
def test_sigmoid(hip, M, N, K):
    g = np.random.default_rng(M)
    x, w = g.standard_normal((M, K)).astype(np.float32), (g.standard_normal((K, N)) * K ** -0.5).astype(np.float32)
    (got,) = vectors.run(hip, product(2, False, True), 1, x, w)
    exact = 1 / (1 + np.exp(-(x.astype(np.float64) @ w.astype(np.float64))))
    # (terms of size K^-1/2: their sums are off by 4 sqrt(K) 2^-24 of K^1/2 K^-1/2 at most; f32 exp and division: 4 units)
    assert np.abs(got - exact).max() <= 0.25 * 4 * np.sqrt(K) * 2.0 ** -24 + 4 * 2.0 ** -24


# heights of an odd number of 16 rows: their last rows, the first past them, columns that end in either half of a wavefront's 32, a last
# step of one piece, slices of k, a batch (test_kernel_choice.py asserts the heights)
ODD_SIZES = [(1, 1, 33, 2048, 4100), (1, 1, 48, 4108, 1000), (2, 1, 65, 5380, 1404), (2, 1, 79, 4100, 2060), (3, 1, 97, 4100, 2060), (3, 2, 112, 2068, 1028),
             (4, 1, 144, 2052, 4100), (5, 1, 175, 8196, 2060), (6, 1, 207, 5380, 1404), (7, 1, 225, 5380, 1404), (7, 1, 240, 5380, 1404)]


@pytest.mark.gpu
@pytest.mark.parametrize("along_k", [True, False])
@pytest.mark.parametrize("rows,B,M,N,K", ODD_SIZES)
def test_product_of_an_odd_height(hip, rows, B, M, N, K, along_k):
    test_product(hip, rows, B, M, N, K, along_k)


@pytest.mark.gpu
@pytest.mark.parametrize("along_k", [True, False])
@pytest.mark.parametrize("rows,B,M,N,K", [s for s in ODD_SIZES if s[2] * s[3] < 1e6])
def test_infinities_of_an_odd_height(hip, rows, B, M, N, K, along_k):
    test_infinities(hip, rows, B, M, N, K, along_k)
