"""bf16 products whose main loop is one statement of assembly (gemm_bf16_ring_kernel, mfma_step_ring.hpp): the fewest k-steps
each takes, an odd number, many; rows and columns that end inside a tile and rows of a length that is no multiple of 16 bytes;
the stacked gate / up form with either activation; grouped products with and without a bias, and rotated; a sigmoid stored as
the next product's operand."""
import numpy as np
import pytest

import parity
import test_llama_parity as llama_tests
import test_moe_gemma_parity as moe_tests
import vectors
from test_f32_tiles import assert_infinities, with_infinities

lang, nn, helpers = vectors.cg.lang, vectors.cg.nn, moe_tests.llm.helpers


def draw(g, shape, std=1.0):
    return vectors.bf16_round((g.standard_normal(shape) * std).astype(np.float32))


def linear(b, x, w, n, k, bias=None):
    y = lang.matmul(b, x, lang.reshape(b, lang.make_shape(b, 1, k, n), lang.transpose(b, 0, 1, w)))
    return y if bias is None else y + lang.broadcast(b, bias, lang.shape(b, y))


def product_and_bound(x, w):
    """x w^T in 64 bits and what K f32 additions of exact bf16 products may be off by."""
    x, w = x.astype(np.float64), w.astype(np.float64)
    return x @ w.T, x.shape[-1] * 2.0 ** -24 * (np.abs(x) @ np.abs(w).T)


# 256 x 256 tiles and smaller ones; then 128 x 128 in one round of 33 and 17 steps and in two rounds, 192 x 128 in one round of 4, 5
# and 32 steps and in two rounds
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(4096, 4096, 128), (4097, 4101, 192), (3841, 4353, 256), (8300, 2049, 320), (255, 65600, 448),
                                   (1500, 2050, 2112), (1400, 1410, 1088), (3100, 2050, 4160),
                                   (2300, 2050, 256), (2303, 2049, 320), (2305, 2048, 2048), (4200, 2050, 4096),
                                   (2305, 2049, 64), (2303, 2049, 576), (2303, 2049, 640),    # ... of one and nine steps on eight wavefronts, of ten on four
                                   (140, 700, 192), (300, 300, 256), (1000, 1100, 256),       # less than a round: halves and quarters of 128 x 128
                                   # 256 x 256 again, with one to three columns in the last piece and quadrants past both edges
                                   (4090, 4093, 192), (3841, 3843, 256), (8001, 2046, 320), (255, 65299, 448), (4096, 4093, 384), (3841, 3843, 576), (8191, 4095, 512)])
def test_product(hip_bf16, M, N, K):
    g = np.random.default_rng(M)
    x, w = draw(g, (1, M, K)), draw(g, (N, K))
    (got,) = vectors.run(hip_bf16, lambda b, x, w: [linear(b, x, w, N, K)], 1, x, w)
    ref, bound = product_and_bound(x[0], w)
    assert np.all(np.abs(got[0] - ref) <= bound)


# 256 x 288: one round where 256 x 256 take two, the fewest k-steps it is given, an odd number; rows that end in the first and the second
# half of a tile, columns that end in the strip and in front of it; and less than a round of 256 x 256 in place of two of 128 x 128
# (test_kernel_choice.py holds these lists, and those of tiles that rotate, to the kernel they are meant for)
WIDE = [(4100, 4308, 256), (4250, 4084, 320), (4352, 4320, 576), (3900, 4148, 1088)]
NOT_WIDE = [(3001, 3003, 768), (2100, 4100, 1024)]


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", WIDE + NOT_WIDE)
def test_wide_product(hip_bf16, M, N, K):
    test_product(hip_bf16, M, N, K)


WIDE_BATCH = (3, 1300, 4028, 256)


@pytest.mark.gpu
@pytest.mark.parametrize("B,M,N,K", [(1, *WIDE[0]), (1, *WIDE[1]), WIDE_BATCH, (1, *NOT_WIDE[0])])
def test_wide_product_and_residual(hip_bf16, B, M, N, K):
    test_product_and_residual(hip_bf16, B, M, N, K)


WIDE_GATED = [(4100, 2152, 256), (4250, 2056, 320), (3900, 2304, 640)]    # columns that end in the strip, in front of it, with a tile


@pytest.mark.gpu
@pytest.mark.parametrize("act", ["silu", "gelu"])
@pytest.mark.parametrize("M,F,K", WIDE_GATED)
def test_wide_gated(hip_bf16, M, F, K, act):
    test_gated(hip_bf16, M, F, K, act)


@pytest.mark.gpu
def test_wide_infinities(hip_bf16):
    test_infinities(hip_bf16, 4100, 4308, 256)


# one column (a wave to a row, its last pieces of k partly past the end, or 64 x 64 tiles), and more than 32 columns but less than 64:
# tiles of 32 x 32 and of 64 x 64 at both ends of either, slices of the deepest
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1030, 1, 2048), (17, 1, 200), (300, 1, 2056), (65, 1, 8), (17, 1, 72), (6001, 1, 176), (6001, 1, 192), (16385, 1, 504),
                                   (1030, 60, 2048), (65, 33, 64), (129, 63, 1088), (9, 60, 1024), (200, 60, 4096), (200, 60, 4160),
                                   (65, 33, 384), (65, 33, 448), (513, 61, 320), (8192, 60, 448), (8193, 60, 512), (1023, 63, 4096), (3072, 60, 4096)])
def test_narrow_product(hip_bf16, M, N, K):
    test_product(hip_bf16, M, N, K)


# 256 x 256 on four and eight wavefronts, 192 x 128 and 128 x 128 on four, their quarters, a wave to a row, 32 x 32, copied operands
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(3841, 3843, 576), (4090, 4093, 192), (2303, 2049, 640), (1400, 1410, 1088), (300, 300, 256),
                                   (1030, 1, 2048), (129, 63, 1088), (900, 1100, 1000)])
def test_infinities(hip_bf16, M, N, K):
    g = np.random.default_rng(M)
    x, w = with_infinities(draw(g, (M, K)), draw(g, (N, K)))
    (got,) = vectors.run(hip_bf16, lambda b, x, w: [linear(b, x, w, N, K)], 1, x[None], w)
    assert_infinities(x, w, got[0])


# a residual added as the product is stored: each tile that does so, whole rounds of large tiles with the rest on smaller ones
# (also where the rounds alone would leave 40 rows), quadrants of a tile past every edge and three columns in the last piece, a batch, and the forms that leave the add to someone else (64 rows, k-slices)
@pytest.mark.gpu
@pytest.mark.parametrize("B,M,N,K", [(1, 4097, 4101, 192), (1, 8300, 2050, 2048), (1, 1500, 2050, 2112), (1, 2303, 2049, 320), (1, 2303, 2049, 640), (1, 3100, 2050, 1024),
                                     (1, 8232, 2048, 2048), (1, 296, 33000, 2048), (1, 3300, 2050, 2048),
                                     (1, 3841, 3843, 128), (1, 4090, 4093, 192), (1, 8001, 2046, 256), (16, 1000, 1002, 128), (1, 300, 130, 64), (1, 1000, 1000, 256), (3, 700, 520, 192), (1, 64, 200, 128),
                                     (1, 200, 300, 2048), (1, 4816, 35, 3648), (1, 17, 60, 320), (3, 700, 61, 512)])    # (the last three: 32 x 32 tiles)
def test_product_and_residual(hip_bf16, B, M, N, K):
    g = np.random.default_rng(M)
    x, w, r = draw(g, (B, M, K)), draw(g, (N, K) if B == 1 else (B, N, K)), draw(g, (B, M, N), 3.0)

    def f(b, x, w, r):
        r = r + r - r       # (f32, like a stream of residuals, and read by others too)
        return [r + (linear(b, x, w, N, K) if B == 1 else lang.matmul(b, x, lang.transpose(b, 1, 2, w))), r]
    hip_bf16.launch_counts(reset=True)
    got, _ = vectors.run(hip_bf16, f, 2, x, w, r)
    counts = hip_bf16.launch_counts(reset=True)
    assert counts.get("gemm") == 1 and counts.get("ew_fused") == 1 and (M <= 64 <= N) == ("binary_f32" in counts), counts     # (ew_fused: r)
    for i in range(B):
        ref, bound = product_and_bound(x[i], w if B == 1 else w[i])
        ref = ref + r[i]
        assert np.all(np.abs(got[i] - ref) <= bound + 2.0 ** -24 * (np.abs(ref) + bound))


@pytest.mark.gpu
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("M,K", [(21900, 128), (22016, 192)])
def test_grouped_products(hip_bf16, M, K, bias):
    g = np.random.default_rng(K)
    x, ws, bs = draw(g, (1, M, K)), [draw(g, (256, K)) for _ in range(3)], [g.standard_normal(256).astype(np.float32) for _ in range(3)]

    def f(b, x, *p):
        return [linear(b, x, p[i], 256, K, p[3 + i] if bias else None) for i in range(3)]
    got = vectors.run(hip_bf16, f, 3, x, *ws, *bs)
    for w, v, y in zip(ws, bs, got):
        ref, bound = product_and_bound(x[0], w)
        if bias:    # one more f32 addition
            ref, bound = ref + v, bound + 2.0 ** -24 * (np.abs(ref) + np.abs(v))
        assert np.all(np.abs(y[0] - ref) <= bound)


@pytest.mark.gpu
@pytest.mark.parametrize("act", ["silu", "gelu"])
@pytest.mark.parametrize("M,F,K", [(4096, 2048, 128), (4100, 2056, 192), (3900, 2184, 320),    # tiles of 256 rows
                                   (1030, 2184, 192), (900, 3000, 256), (1000, 2824, 512),     # and of 128: three steps, four, more
                                   (4100, 2056, 64), (4200, 2600, 128), (4100, 1256, 128), (1000, 3000, 64), (1030, 2184, 128),    # one and two, on eight wavefronts or four
                                   (700, 8192, 512), (577, 7688, 576), (768, 6920, 640), (1153, 8200, 512),    # of 192: eight steps, nine, ten; two rounds
                                   (4100, 2052, 192), (1030, 2180, 192), (1000, 2820, 512)])   # two products: rows of results off 16 bytes
def test_gated(hip_bf16, M, F, K, act):
    g = np.random.default_rng(F)
    x, wg, wu, wd = draw(g, (1, M, K)), draw(g, (F, K), K ** -0.5), draw(g, (F, K), K ** -0.5), np.eye(64, F, dtype=np.float32)

    def f(b, x, wg, wu, wd):    # (wd picks the first 64 gated values out: exact products)
        x = x + x - x
        return [linear(b, getattr(nn, act)(b, linear(b, x, wg, F, K)) * linear(b, x, wu, F, K), wd, 64, F)]
    hip_bf16.launch_counts(reset=True)
    (got,) = vectors.run(hip_bf16, f, 1, x, wg, wu, np.roll(wd, F - 64, axis=1))
    counts = hip_bf16.launch_counts(reset=True)
    assert counts.get("gemm") == (3 if F % 8 else 2), counts
    gate, up = (x[0].astype(np.float64) @ w[F - 64:].astype(np.float64).T for w in (wg, wu))
    c = gate if act == "silu" else 2 * np.sqrt(2 / np.pi) * (gate + 0.044715 * gate ** 3)
    ref = gate / (1 + np.exp(-c)) * up
    # rounded once to bf16, whose eight significant bits leave half a unit in the last place: 2^-8 of the value at most, and 2^-19 for
    # the hardware's exp2 and reciprocal; the f32 sums in front of it, of K terms of size K^-1/2, are off by 4 sqrt(K) 2^-24 at most
    # (as in assert_f32_sums), and no slope of an activation is above 1.13
    sums = 4 * np.sqrt(K) * 2.0 ** -24 * (1.13 * np.abs(up) + np.abs(gate))
    assert np.all(np.abs(got[0] - ref) <= (2.0 ** -8 + 2.0 ** -19) * np.abs(ref) + sums)


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,H", [(4100, 130, 4099), (4352, 192, 3900)])
def test_sigmoid_as_the_next_operand(hip_bf16, M, K, H):
    g = np.random.default_rng(H)
    x, w1 = draw(g, (M, K)), draw(g, (K, H), K ** -0.5)
    w2 = np.zeros((H, 64), np.float32)
    w2[H - 64 + np.arange(64), np.arange(64)] = 1.0
    (got,) = vectors.run(hip_bf16, lambda b, x, w1, w2: [lang.matmul(b, nn.sigmoid(b, lang.matmul(b, x, w1)), w2)], 1, x, w1, w2)
    ref = 1 / (1 + np.exp(-(x.astype(np.float64) @ w1[:, H - 64:].astype(np.float64))))
    assert np.all(np.abs(got - ref) <= 2.0 ** -8 * ref + 1e-5)    # (as above)


# less than a round of tiles that rotate, one, more than one, heads of 64 and of 128, with and without biases, several
# sequences, positions in no multiple of four
@pytest.mark.gpu
@pytest.mark.parametrize("tokens", [1601, 318, 130])
def test_rotated(oracle, hip_bf16, tokens):
    llama_tests.test_llama_prefill_rotates_in_the_projections_launch(oracle, hip_bf16, tokens, 16, 16, 1)


@pytest.mark.gpu
@pytest.mark.parametrize("batch,tokens", [(2, 301), (3, 550), (1, 317), (2, 65)])
def test_rotated_wide_heads(oracle, hip_bf16, batch, tokens):
    moe_tests.test_qwen_prefill_biases_and_rotation_in_the_projections_launch(oracle, hip_bf16, batch, tokens, 8, 8, 128)


# q / k / v that leave a 256 x 256 tile rotated: heads of 64, 128 and 256, with biases, with a norm of every head's row in front of the
# rotation; one sequence that ends inside a tile, several whose length is no multiple of four (pieces of values that straddle two), of eight
ROTATED_LARGE = [(64, 1, 2203, 20, 20, 768, False, False), (64, 8, 276, 20, 20, 768, True, False),
                 (128, 5, 271, 16, 16, 768, True, False), (128, 1, 1302, 16, 16, 832, False, False),
                 (256, 21, 257, 4, 1, 192, False, True), (256, 129, 64, 2, 1, 128, False, True),
                 (256, 20, 270, 4, 1, 128, False, False)]


def attention_of_projections(b, x, p, hd, batch, S, heads, kv, K, bias, norm, eps=1e-6, theta=10000.0):
    """Attention, rotated keys and values of x; p: the three weights, their biases, the gammas of queries and keys (none: no gamma)."""
    h, ns = helpers, [heads * hd, kv * hd, kv * hd]

    def normed(gamma, n_heads, y):   # (gemma3.rs:41-68, folded as in gemma3.rs:99-117)
        y = lang.reshape(b, lang.make_shape(b, batch * n_heads * S, hd), y)
        s = lang.sum(b, y * y)
        mean = s / lang.broadcast(b, lang.cast(b, lang.nat_to_u32(b, lang.to_nat(b, hd)), lang.dtype(b, y)), lang.shape(b, s))
        rms = nn.sqrt(b, mean + lang.constant(b, eps, lang.shape(b, mean)))
        y = y / lang.broadcast(b, rms, lang.shape(b, y))
        if gamma is not None:
            gm = lang.broadcast(b, gamma, lang.shape(b, y))
            y = y * (lang.constant(b, 1.0, lang.shape(b, gm)) + gm)
        return lang.reshape(b, lang.make_shape(b, batch, n_heads, S, hd), y)

    y = [linear(b, x, p[i], ns[i], K, p[3 + i] if bias else None) for i in range(3)]
    y = [lang.transpose(b, 1, 2, lang.reshape(b, lang.make_shape(b, batch, S, n // hd, hd), t)) for n, t in zip(ns, y)]
    gammas = p[6:8] if len(p) > 6 else [None, None]
    q, k, v = y if not norm else [normed(gammas[0], heads, y[0]), normed(gammas[1], kv, y[1]), y[2]]
    q, k = h.rope(b, theta, 0, S, hd, q), h.rope(b, theta, 0, S, hd, k)
    attn = lang.matmul(b, q, lang.transpose(b, 2, 3, h.repeat_kv(b, heads // kv, k)))
    sh = lang.shape(b, attn)
    attn = attn / lang.constant(b, float(np.sqrt(np.float32(hd))), sh) + lang.broadcast(b, h.causal_mask(b, lang.to_nat(b, S)), sh)
    return [lang.matmul(b, nn.softmax(b, attn), h.repeat_kv(b, heads // kv, v)), k, v]


@pytest.mark.gpu
@pytest.mark.parametrize("hd,batch,S,heads,kv,K,bias,norm", ROTATED_LARGE)
def test_rotated_on_large_tiles(hip_bf16, hd, batch, S, heads, kv, K, bias, norm):
    g = np.random.default_rng(S)
    x, ns = draw(g, (1, batch * S, K)), [heads * hd, kv * hd, kv * hd]
    ws, bs = [draw(g, (n, K), K ** -0.5) for n in ns], [g.standard_normal(n).astype(np.float32) for n in ns]
    gammas = [(0.3 * g.standard_normal(hd)).astype(np.float32) for _ in range(2)]
    h, theta, eps = helpers, 10000.0, 1e-6

    def f(b, x, *p):
        return attention_of_projections(b, x + x - x, p, hd, batch, S, heads, kv, K, bias, norm, eps, theta)
    hip_bf16.trace(2)
    hip_bf16.trace_reset()
    got, k, v = vectors.run(hip_bf16, f, 3, x, *ws, *bs, *gammas)
    names = sorted(hip_bf16.trace_report())
    hip_bf16.trace(False)
    assert sum("grouped,rope" in n for n in names) == 1 and not any(n.startswith(("rope_fused", "transpose_cast_bf16")) for n in names), names
    c, s = (t.astype(np.float64) for t in vectors.run(hip_bf16, lambda b, _: h.rope_tables(b, theta, lang.to_nat(b, S), hd), 2, np.zeros(1, np.float32)))
    y = [x[0].astype(np.float64) @ w.T.astype(np.float64) + (v64 if bias else 0.0) for w, v64 in zip(ws, bs)]
    y = [t.reshape(batch, S, -1, hd).transpose(0, 2, 1, 3) for t in y]
    if norm:
        for i in range(2):
            y[i] = y[i] / np.sqrt(np.mean(y[i] ** 2, axis=-1, keepdims=True) + eps) * (1.0 + gammas[i].astype(np.float64))
    for i in range(2):
        y[i] = c * y[i] + s * np.concatenate([-y[i][..., hd // 2:], y[i][..., :hd // 2]], axis=-1)
    parity.assert_f32(y[1], k, "rotated keys")
    parity.assert_f32(y[2], v, "values")
    keys, values = (np.repeat(t, heads // kv, axis=1).astype(np.float32) for t in y[1:])
    scores = (y[0].astype(np.float32) @ keys.transpose(0, 1, 3, 2)) / np.sqrt(np.float32(hd))
    scores = np.where(np.tri(S, dtype=bool), scores, -np.inf)
    scores = np.exp(scores - scores.max(axis=-1, keepdims=True))
    parity.assert_bf16((scores / scores.sum(axis=-1, keepdims=True)) @ values, got, "attention")


# ... (of those, the heads of 64 and of 128 above are in one round of 192 x 256; here, in none)
ROTATED_256 = [(64, 1, 3301, 20, 20, 768, False, False), (64, 12, 277, 20, 20, 832, True, False),
               (128, 7, 279, 16, 16, 768, True, False), (128, 1, 1930, 16, 16, 832, False, False)]


@pytest.mark.gpu
@pytest.mark.parametrize("hd,batch,S,heads,kv,K,bias,norm", ROTATED_256)
def test_rotated_on_256_rows(hip_bf16, hd, batch, S, heads, kv, K, bias, norm):
    test_rotated_on_large_tiles(hip_bf16, hd, batch, S, heads, kv, K, bias, norm)


# ... and on tiles of 128 x 256, where those are one round
ROTATED_HALF = [(64, 1, 1203, 20, 20, 768, False, False), (64, 6, 203, 20, 20, 832, True, False),
                (128, 5, 151, 16, 16, 768, True, False), (128, 1, 1202, 16, 16, 832, False, False),
                (256, 11, 257, 4, 1, 768, False, True), (256, 45, 64, 4, 1, 832, False, True),
                (256, 11, 270, 4, 1, 768, False, False)]


@pytest.mark.gpu
@pytest.mark.parametrize("hd,batch,S,heads,kv,K,bias,norm", ROTATED_HALF)
def test_rotated_on_half_tiles(hip_bf16, hd, batch, S, heads, kv, K, bias, norm):
    test_rotated_on_large_tiles(hip_bf16, hd, batch, S, heads, kv, K, bias, norm)


# ... the norm in front of the rotation on rows that it treats specially, with gamma and without: zeros, values whose squares vanish or
# overflow (the quotient by infinity is 0), infinities and a NaN (the quotient is none), beside rows of neither kind
@pytest.mark.gpu
@pytest.mark.parametrize("gamma", [True, False])
@pytest.mark.parametrize("batch,S,K", [(21, 257, 192), (11, 257, 768)])
def test_special_rows_normed_and_rotated(hip_bf16, batch, S, K, gamma):
    g, hd, heads, eps, theta = np.random.default_rng(S + K), 256, 4, 1e-6, 10000.0
    x = draw(g, (1, batch * S, K))
    rows = g.permutation(batch * S)[:30].reshape(6, 5)      # (any place of a tile and of a wavefront's rows)
    x[0, rows[0]] = 0.0
    x[0, rows[1]] *= np.float32(2.0 ** -80)
    x[0, rows[2]] *= np.float32(2.0 ** 70)
    x[0, rows[3], 0] = np.inf
    x[0, rows[4], K - 1] = -np.inf
    x[0, rows[5], 1] = np.nan
    ns = [heads * hd, hd, hd]
    ws, bs = [draw(g, (n, K), K ** -0.5) for n in ns], [np.zeros(n, np.float32) for n in ns]
    ws[1][:, [0, K - 1]] = np.where(ws[1][:, [0, K - 1]] == 0, np.float32(0.5), ws[1][:, [0, K - 1]])
    gammas = [(0.3 * g.standard_normal(hd)).astype(np.float32) for _ in range(2)] if gamma else []
    hip_bf16.trace(2)
    hip_bf16.trace_reset()
    def f(b, x, *p):
        x = x * lang.constant(b, 1.0, lang.shape(b, x))     # (f32, and infinities stay)
        return attention_of_projections(b, x, p, hd, batch, S, heads, 1, K, False, True, eps, theta)
    _, k, _ = vectors.run(hip_bf16, f, 3, x, *ws, *bs, *gammas)
    names = sorted(hip_bf16.trace_report())
    hip_bf16.trace(False)
    assert sum("grouped,rope" in n for n in names) == 1 and not any(n.startswith("rope_fused") for n in names), names
    k = k.reshape(batch * S, hd)
    assert np.all(k[rows[[0, 2]].ravel()] == 0) and np.all(np.isnan(k[rows[3:].ravel()]))
    finite = np.setdiff1d(np.arange(batch * S), rows[2:].ravel())
    c, s = (t.astype(np.float64) for t in vectors.run(hip_bf16, lambda b, _: helpers.rope_tables(b, theta, lang.to_nat(b, S), hd), 2, np.zeros(1, np.float32)))
    y = x[0, finite].astype(np.float64) @ ws[1].T.astype(np.float64)
    y = y / np.sqrt(np.mean(y ** 2, axis=-1, keepdims=True) + eps) * (1.0 + gammas[1].astype(np.float64) if gamma else 1.0)
    c, s = (t.reshape(S, hd)[finite % S] for t in (c, s))
    ref = c * y + s * np.concatenate([-y[:, hd // 2:], y[:, :hd // 2]], axis=-1)
    tiny = np.isin(finite, rows[1])     # (on a scale of their own)
    parity.assert_f32(ref[~tiny], k[finite[~tiny]], "rotated keys")
    parity.assert_f32(ref[tiny] * 2.0 ** 80, k[finite[tiny]].astype(np.float64) * 2.0 ** 80, "rotated keys of tiny rows")


# 128 x 256 in one round: the fewest k-steps, an odd number, rows and columns that end inside a tile, rows of results off 16 bytes, a batch
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(3100, 2050, 1024), (3333, 2049, 1088), (2300, 3001, 2048), (1000, 6143, 1152), (4096, 2048, 4160)])
def test_half_height_product(hip_bf16, M, N, K):
    test_product(hip_bf16, M, N, K)


@pytest.mark.gpu
@pytest.mark.parametrize("B,M,N,K", [(1, 3100, 2050, 1024), (1, 4000, 2048, 1088), (2, 1601, 2047, 1024)])
def test_half_height_product_and_residual(hip_bf16, B, M, N, K):
    test_product_and_residual(hip_bf16, B, M, N, K)


@pytest.mark.gpu
def test_half_height_infinities(hip_bf16):
    test_infinities(hip_bf16, 3333, 2049, 1088)


# attention whose result only a product of many rows reads: queries and result as bf16 only.  The product with one is that result, and the
# same bits as the f32 result rounded, which another reader has it store; every form of the kernel, a batch, keys that end inside a tile
@pytest.mark.gpu
@pytest.mark.parametrize("hd,batch,S,heads,kv", [(64, 1, 100, 8, 2), (64, 1, 512, 8, 2), (64, 1, 1502, 8, 2), (64, 1, 2903, 8, 2), (64, 3, 70, 8, 8), (128, 2, 700, 8, 4),
                                                 (128, 1, 3000, 8, 4), (128, 4, 256, 16, 8), (256, 8, 1000, 4, 1), (256, 1, 703, 4, 1), (256, 2, 100, 4, 1)])
def test_attention_read_by_a_product(hip_bf16, hd, batch, S, heads, kv):
    g, K, h = np.random.default_rng(S), 192, helpers
    ns = [heads * hd, kv * hd, kv * hd]
    x, ws, eye = draw(g, (1, batch * S, K)), [draw(g, (n, K), K ** -0.5) for n in ns], np.eye(heads * hd, dtype=np.float32)

    def f(b, x, *p, also):
        x = x + x - x
        y = [linear(b, x, w, n, K) for w, n in zip(p, ns)]
        q, k, v = (lang.transpose(b, 1, 2, lang.reshape(b, lang.make_shape(b, batch, S, n // hd, hd), t)) for n, t in zip(ns, y))
        q, k = h.rope(b, 10000.0, 0, S, hd, q), h.rope(b, 10000.0, 0, S, hd, k)
        attn = lang.matmul(b, q, lang.transpose(b, 2, 3, h.repeat_kv(b, heads // kv, k)))
        sh = lang.shape(b, attn)
        attn = attn / lang.constant(b, float(np.sqrt(np.float32(hd))), sh) + lang.broadcast(b, h.causal_mask(b, lang.to_nat(b, S)), sh)
        out = lang.matmul(b, nn.softmax(b, attn), h.repeat_kv(b, heads // kv, v))
        merged = lang.reshape(b, lang.make_shape(b, 1, batch * S, ns[0]), lang.transpose(b, 1, 2, out))
        return [linear(b, merged, p[3], ns[0], ns[0])] + ([out] if also else [])

    def run(also):
        hip_bf16.trace(2)
        hip_bf16.trace_reset()
        got = vectors.run(hip_bf16, lambda b, *a: f(b, *a, also=also), 2 if also else 1, x, *ws, eye)
        names = set(hip_bf16.trace_report())
        hip_bf16.trace(False)
        assert ("attn_prefill" if also else "attn_prefill[bf16]") in names, sorted(names)
        return got
    (narrow,), (_, out) = run(False), run(True)
    assert np.array_equal(narrow[0].reshape(batch, S, heads, hd), vectors.bf16_round(out).transpose(0, 2, 1, 3))


# the routed experts of a prefill, from 44 pairs to an expert on moe_ring_kernel: three slots whose choices crowd one expert (several row tiles, the last
# partly filled) and leave others empty; the fewest k-steps, columns that end inside a tile of 128 and of 256; more pairs than
# moe_route_kernel keeps in registers, more experts than it has threads
@pytest.mark.gpu
@pytest.mark.parametrize("act", ["silu", "gelu"])
@pytest.mark.parametrize("S,E,F,H", [(150, 6, 192, 192), (64, 9, 320, 576), (140, 9, 320, 576), (700, 5, 256, 192),
                                     (2800, 5, 64, 64), (300, 1100, 64, 64)])
def test_routed_experts(oracle, hip_bf16, S, E, F, H, act):
    g = np.random.default_rng(S)
    x, k = draw(g, (S, 1, H)), 3
    wg, wu, wd = draw(g, (E, F, H), H ** -0.5), draw(g, (E, F, H), H ** -0.5), draw(g, (E, H, F), F ** -0.5)
    idx = np.where(g.random((S, k)) < 0.6, 2, g.integers(0, E - 1, (S, k))).astype(np.uint32)
    val = g.random((S, k)).astype(np.float32)

    def f(b, x, iv, vv, wg, wu, wd):
        x = x + x - x
        total = None
        for i in range(k):
            slot = lang.get(b, 1, i, iv)
            sel = lambda w: lang.transpose(b, 1, 2, lang.index(b, 0, slot, w))
            y = lang.matmul(b, getattr(nn, act)(b, lang.matmul(b, x, sel(wg))) * lang.matmul(b, x, sel(wu)), sel(wd))
            y = y * lang.broadcast(b, lang.reshape(b, lang.shape(b, lang.get(b, 2, 0, y)), lang.get(b, 1, i, vv)), lang.shape(b, y))
            total = y if total is None else total + y
        return [total]
    (ref,) = vectors.run(oracle, f, 1, x, idx, val, wg, wu, wd)
    (got,) = vectors.run(hip_bf16, f, 1, x, idx, val, wg, wu, wd)
    parity.assert_bf16(ref, got, f"{S} tokens")


# a product of a few dozen columns and one of a single column of the same rows (a MoE layer's router and its shared expert's gate): one
# launch, a tile more; partly filled tiles of rows and columns, the fewest k, and more rows than two workgroups to a CU hold
# (up to 128 rows of 2048 values and more, whose column tiles start at different k, test_k_order.py; weights of a multiple of 4 KB and others)
WITH_COLUMN = [(1024, 60, 2048, True), (17, 60, 1024, True), (33, 34, 448, True), (65, 63, 512, True), (5440, 60, 448, True), (5473, 60, 448, False),
               (20, 60, 2048, True), (128, 63, 2048, True), (90, 33, 2048, True), (128, 60, 2112, True), (129, 60, 2048, True)]


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,joined", WITH_COLUMN)
def test_product_with_a_column(hip_bf16, M, N, K, joined):
    g = np.random.default_rng(M)
    x, w, col = draw(g, (1, M, K)), draw(g, (N, K), K ** -0.5), draw(g, (1, K), K ** -0.5)

    def f(b, x, w, col):
        x = x + x - x
        return [linear(b, x, w, N, K), linear(b, x, col, 1, K)]
    hip_bf16.launch_counts(reset=True)
    got = vectors.run(hip_bf16, f, 2, x, w, col)
    counts = hip_bf16.launch_counts(reset=True)
    assert sum(c for n, c in counts.items() if n.startswith("gem")) == 2 - joined, counts
    for y, weight in zip(got, (w, col)):
        ref, bound = product_and_bound(x[0], weight)
        assert np.all(np.abs(y[0] - ref) <= bound)
