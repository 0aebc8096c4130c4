"""Products of sizes that are no multiple of a tile or of 16 bytes in bf16 mode: operands copied to padded rows for the
direct-to-LDS kernel, from every storage order; and sigmoid(product), stored by the product's launch as f32, as the next
product's bf16 operand, or by the pass that sums the k-slices."""
import numpy as np
import pytest

import parity
import vectors

lang, nn = vectors.cg.lang, vectors.cg.nn


def mlp(b, x, w1, w2):
    return [lang.matmul(b, nn.sigmoid(b, lang.matmul(b, x, w1)), w2)]


def sigmoid_of_product(b, x, w1):
    return [nn.sigmoid(b, lang.matmul(b, x, w1))]


def transposed(b, x, w):   # x [.., k, m], w [.., n, k]
    return [lang.matmul(b, lang.transpose(b, 1, 2, x), lang.transpose(b, 1, 2, w))]


def plain(b, x, w):
    return [lang.matmul(b, x, w)]


def draw(g, shape, std):
    return vectors.bf16_round((g.standard_normal(shape) * std).astype(np.float32))


# below and above the size from which operands are copied; hidden sizes of one value past a tile, of a multiple of 64 and
# with an odd tail; outputs of less than a tile; rows that end inside a tile
SIZES = [(64, 128, 256, 10), (70, 100, 300, 17), (300, 200, 130, 64), (257, 999, 2050, 100), (513, 1000, 1027, 12),
         (1000, 513, 1024, 99), (1030, 64, 8197, 65), (2100, 72, 4100, 10)]


@pytest.mark.gpu
@pytest.mark.parametrize("rows,inner,hidden,outer", SIZES)
@pytest.mark.parametrize("bf16", [True, False])
def test_hidden_layer(oracle, hip, hip_bf16, rows, inner, hidden, outer, bf16):
    g = np.random.default_rng(rows)
    x, w1, w2 = draw(g, (rows, inner), 1.0), draw(g, (inner, hidden), inner ** -0.5), draw(g, (hidden, outer), hidden ** -0.5)
    (ref,) = vectors.run(oracle, mlp, 1, x, w1, w2)
    (got,) = vectors.run(hip_bf16 if bf16 else hip, mlp, 1, x, w1, w2)
    (parity.assert_bf16 if bf16 else parity.assert_f32)(ref, got, f"{rows}x{inner}x{hidden}x{outer}")


@pytest.mark.gpu
@pytest.mark.parametrize("rows,inner,hidden", [(9, 40, 33), (64, 2048, 64), (100, 300, 77), (600, 256, 640), (777, 1001, 905)])
@pytest.mark.parametrize("bf16", [True, False])
def test_sigmoid_of_a_product(oracle, hip, hip_bf16, rows, inner, hidden, bf16):
    g = np.random.default_rng(rows)
    x, w = draw(g, (rows, inner), 1.0), draw(g, (inner, hidden), inner ** -0.5)
    x[0, :] = 200.0 * np.sign(w[:, 0])      # a sum far into both tails
    x[1, :] = -x[0, :]
    (ref,) = vectors.run(oracle, sigmoid_of_product, 1, x, w)
    (got,) = vectors.run(hip_bf16 if bf16 else hip, sigmoid_of_product, 1, x, w)
    (parity.assert_bf16 if bf16 else parity.assert_f32)(ref, got, f"{rows}x{inner}x{hidden}")


# both strides of a single column are 1 as it lies, and the kernels for few k or few rows of it have no sigmoid of their own
@pytest.mark.gpu
@pytest.mark.parametrize("rows,inner", [(9, 16), (64, 64), (65, 64), (100, 200), (6001, 184), (6001, 192), (20, 2048)])
@pytest.mark.parametrize("batch", [1, 3])
def test_sigmoid_of_one_column(oracle, hip_bf16, batch, rows, inner):
    g = np.random.default_rng(rows)
    x, w = draw(g, (batch, rows, inner), 1.0), draw(g, (batch, inner, 1), inner ** -0.5)
    for f, right in ((sigmoid_of_product, w), (lambda b, x, w: [nn.sigmoid(b, lang.matmul(b, x, lang.transpose(b, 1, 2, w)))], w.reshape(batch, 1, inner))):
        (ref,) = vectors.run(oracle, f, 1, x, right)
        (got,) = vectors.run(hip_bf16, f, 1, x, right)
        parity.assert_bf16(ref, got, f"{batch} x {rows} x {inner}")


@pytest.mark.gpu
@pytest.mark.parametrize("batch,m,n,k", [(1, 700, 900, 801), (3, 260, 516, 1002), (2, 1001, 300, 904), (1, 515, 1030, 1024)])
@pytest.mark.parametrize("turned", [True, False])
def test_ragged_operands_of_either_order(oracle, hip_bf16, batch, m, n, k, turned):
    g = np.random.default_rng(m)
    x, w = draw(g, (batch, k, m) if turned else (batch, m, k), 1.0), draw(g, (batch, n, k) if turned else (batch, k, n), k ** -0.5)
    (ref,) = vectors.run(oracle, transposed if turned else plain, 1, x, w)
    (got,) = vectors.run(hip_bf16, transposed if turned else plain, 1, x, w)
    parity.assert_bf16(ref, got, f"{batch}x{m}x{n}x{k}")


# as many 128-row tiles as need a second round over the CUs, and few enough tiles of 192 rows for one; rows and columns that end
# inside a tile, k of one step and of several
@pytest.mark.gpu
@pytest.mark.parametrize("rows,n,k", [(2300, 2048, 64), (2881, 1990, 192), (3071, 1920, 256), (193 * 16, 1536, 128)])
def test_one_round_of_tall_tiles(oracle, hip_bf16, rows, n, k):
    g = np.random.default_rng(rows)
    x, w = draw(g, (1, rows, k), 1.0), draw(g, (1, n, k), k ** -0.5)

    def f(b, x, w):
        return [lang.matmul(b, x, lang.transpose(b, 1, 2, w))]
    (ref,) = vectors.run(oracle, f, 1, x, w)
    (got,) = vectors.run(hip_bf16, f, 1, x, w)
    parity.assert_bf16(ref, got, f"{rows}x{n}x{k}")


# f32 rows rounded to bf16 on their way into a product: every upper half of a finite normal number, with lower halves around a tie, a
# row to each sign and exponent; a product with the unit matrix returns what they became
@pytest.mark.gpu
@pytest.mark.parametrize("lower", [0x0000, 0x0001, 0x7FFF, 0x8000, 0x8001, 0xFFFF])
def test_rounding_of_rows(hip_bf16, lower):
    upper = np.arange(1 << 16, dtype=np.uint32).reshape(-1, 128)
    upper = upper[((upper[:, 0] >> 7 & 255) > 0) & ((upper[:, 0] >> 7 & 255) < 254)]
    x = (upper << 16 | lower).view(np.float32)
    rows = x.shape[0]
    (got,) = vectors.run(hip_bf16, lambda b, x, w: [lang.matmul(b, lang.reshape(b, lang.make_shape(b, rows, 128), x), w)], 1, x.ravel(), np.eye(128, dtype=np.float32))
    assert np.array_equal(got, vectors.bf16_round(x))


# 1 to 8 rows: bf16 rows in slices of k, f32 rows a few steps of k at a time; columns that end inside a piece and inside 64, k off every
# step, infinities at either end of k
@pytest.mark.gpu
@pytest.mark.parametrize("M,K,H,N", [(1, 1073, 743, 69), (5, 1073, 743, 69), (8, 257, 130, 65), (2, 63, 66, 3), (7, 2048, 515, 10), (3, 129, 64, 64)])
@pytest.mark.parametrize("mode", ["hip", "hip_bf16"])
def test_a_few_ragged_rows(request, mode, M, K, H, N):
    be, g = request.getfixturevalue(mode), np.random.default_rng(M * K)
    rounded = lambda s, std: vectors.bf16_round((g.standard_normal(s) * std).astype(np.float32))
    x, w1, w2 = rounded((M, K), 1.0), rounded((K, H), K ** -0.5), rounded((H, N), H ** -0.5)
    y, h = vectors.run(be, lambda b, x, w1, w2: [lang.matmul(b, lang.matmul(b, x, w1) * lang.matmul(b, x, w1), w2), lang.matmul(b, x, w1)], 2, x, w1, w2)
    x64, w64 = x.astype(np.float64), w1.astype(np.float64)
    ref, bound = x64 @ w64, K * 2.0 ** -24 * (np.abs(x64) @ np.abs(w64))     # K f32 additions of exact products
    assert np.all(np.abs(h - ref) <= bound)
    rows = (h * h).astype(np.float64)
    # (f32 rows as they are, or rounded to bf16 where the product does that)
    bound = ((2.0 ** -8 if be.name.startswith("hip") and mode == "hip_bf16" else 0) + (H + 1) * 2.0 ** -24) * (rows @ np.abs(w2.astype(np.float64)))
    assert np.all(np.abs(y - rows @ w2.astype(np.float64)) <= bound)
    x[0, 0], x[-1, -1] = np.inf, np.nan
    (h,) = vectors.run(be, lambda b, x, w1: [lang.matmul(b, x, w1)], 1, x, w1)
    with np.errstate(invalid="ignore"):
        ref = x.astype(np.float64) @ w64
    assert np.array_equal(np.isnan(h), np.isnan(ref)) and np.array_equal(np.isinf(h), np.isinf(ref))


# 2 to 8 f32 rows against k-major weights in slices of k: one slice and the first two, the last one short, some empty; sums that do and do
# not fill pieces of 16 bytes; batches, and a residual that starts on one or off
@pytest.mark.gpu
@pytest.mark.parametrize("batch,M,K,N", [(1, 5, 511, 7), (1, 5, 512, 7), (1, 3, 4112, 5), (1, 8, 1100, 130), (3, 2, 1073, 66), (2, 7, 5000, 1), (40, 4, 600, 64)])
@pytest.mark.parametrize("mode", ["hip", "hip_bf16"])
@pytest.mark.parametrize("residual", [None, 0, 1])
def test_a_few_rows_in_slices_of_k(request, mode, residual, batch, M, K, N):
    be, g = request.getfixturevalue(mode), np.random.default_rng(K)
    rounded = lambda s, std: vectors.bf16_round((g.standard_normal(s) * std).astype(np.float32))
    x, w, r = rounded((batch, M, K), 1.0), rounded((batch, K, N), K ** -0.5), rounded((batch * M * N + 1,), 1.0)
    if residual is not None:
        f = lambda b, x, w, r: [lang.reshape(b, lang.make_shape(b, batch, M, N), lang.slice(b, 0, residual, batch * M * N, r)) + lang.matmul(b, x, w)]
        (y,) = vectors.run(be, f, 1, x, w, r)
    else:
        (y,) = vectors.run(be, plain, 1, x, w)
    x64, w64 = x.astype(np.float64), w.astype(np.float64)
    add = 0.0 if residual is None else r[residual:][:batch * M * N].reshape(batch, M, N).astype(np.float64)
    # K f32 additions of exact products, and one of the residual
    assert np.all(np.abs(y - (x64 @ w64 + add)) <= (K + 1) * 2.0 ** -24 * (np.abs(x64) @ np.abs(w64) + np.abs(add)))
