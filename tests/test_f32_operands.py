"""bf16 mode: which products keep f32 operands beside the bf16 weights.  Their results are held against 64-bit sums with the
tolerance of f32 arithmetic, which an operand rounded to bf16 (2^-9 of each value) misses by two orders of magnitude."""
import importlib

import numpy as np
import pytest

import vectors

lang, nn = vectors.cg.lang, vectors.cg.nn
llm = importlib.import_module("catgrad-rs_amd.llm")
helpers = llm.helpers


def assert_f32_sums(exact, got, terms, what):
    """A sum of n terms in f32: the rounding errors of its additions walk, sqrt(n) * 2^-24 of the terms' root mean square
    sum at most a few times over; the norm of a row against the norm of its exact value."""
    exact, got = (np.asarray(a, np.float64).reshape(-1, np.shape(exact)[-1]) for a in (exact, got))
    err = np.linalg.norm(got - exact, axis=1) / np.linalg.norm(exact, axis=1)
    assert err.max() <= 4 * np.sqrt(terms) * 2.0 ** -24, f"{what}: {err.max():.2e} off"


# 5 to 8 rows at depths beyond the few-row kernel's
@pytest.mark.gpu
@pytest.mark.parametrize("rows", [5, 8])
@pytest.mark.parametrize("K,N", [(4096, 2048), (8192, 2048), (5632, 136), (4096, 65), (4160, 16500), (4100, 128)])
def test_few_rows_of_a_deep_product(hip_bf16, rows, K, N):
    g = np.random.default_rng(rows + K)
    x = g.standard_normal(rows * K).astype(np.float32)
    x[:K] *= np.float32(1e-25)
    x[K:2 * K] *= np.float32(1e30)
    w = vectors.bf16_round((g.standard_normal((N, K)) * K ** -0.5).astype(np.float32))

    def f(b, x, w):
        x = lang.reshape(b, lang.make_shape(b, 1, rows, K), x)     # (uploaded as a vector: f32)
        return [lang.matmul(b, x, lang.reshape(b, lang.make_shape(b, 1, K, N), lang.transpose(b, 0, 1, w)))]
    (got,) = vectors.run(hip_bf16, f, 1, x, w)
    exact = x.reshape(rows, K).astype(np.float64) @ w.astype(np.float64).T
    assert_f32_sums(exact, got, K, f"{rows} x {K} x {N}")

    def k_major(b, x, w):
        return [lang.matmul(b, lang.reshape(b, lang.make_shape(b, rows, K), x), w)]
    (got,) = vectors.run(hip_bf16, k_major, 1, x, np.ascontiguousarray(w.T))
    assert_f32_sums(exact, got, K, f"{rows} x {K} x {N}, k-major")


@pytest.mark.gpu
def test_few_rows_of_a_deep_product_with_a_residual_and_special_values(hip_bf16):
    rows, K, N = 6, 4096, 256
    g = np.random.default_rng(3)
    x, res = (g.standard_normal((rows, n)).astype(np.float32) for n in (K, N))
    w = vectors.bf16_round((g.standard_normal((N, K)) * K ** -0.5).astype(np.float32))
    w[:, 9] = np.where(w[:, 9] == 0, 1, np.abs(w[:, 9]))
    w[5, 9] = 0
    x[0, 9] = np.inf
    x[1, 9] = -np.inf
    x[2].view(np.uint32)[9] = 0x7F800001      # a NaN that only its last bits tell from an infinity
    x[3, 9] = np.finfo(np.float32).max
    x[4] = 0

    def f(b, x, res, w):
        x, res = (lang.reshape(b, lang.make_shape(b, 1, rows, n), t) for t, n in ((x, K), (res, N)))
        y = lang.matmul(b, x, lang.reshape(b, lang.make_shape(b, 1, K, N), lang.transpose(b, 0, 1, w)))
        return [res + y]
    (got,) = vectors.run(hip_bf16, f, 1, x.reshape(-1), res.reshape(-1), w)
    with np.errstate(invalid="ignore"):
        exact = x.astype(np.float64) @ w.astype(np.float64).T + res
    got = got.reshape(rows, N)
    for kind in (np.isposinf, np.isneginf, np.isnan):
        assert np.array_equal(kind(exact), kind(got.astype(np.float64)))
    assert_f32_sums(exact[3:], got[3:], K, "finite rows")


# A few queries: the scores, their exponentials and both products of the attention in f32
@pytest.mark.gpu
@pytest.mark.parametrize("S", [2, 3, 7, 8])
@pytest.mark.parametrize("H,KV,d,T,causal", [(8, 2, 64, 0, True), (4, 4, 128, 0, True), (4, 1, 256, 0, True), (8, 2, 64, 61, False),
                                             (8, 2, 64, 65, False), (2, 2, 128, 32, False), (2, 2, 128, 33, False), (4, 1, 64, 700, False)])
def test_attention_of_a_few_queries(hip_bf16, S, H, KV, d, T, causal):
    T = T or S
    g = np.random.default_rng(S + T)
    q, k, v = (g.standard_normal((h, n, d)).astype(np.float32) for h, n in ((H, S), (KV, T), (KV, T)))

    def f(b, q, k, v):
        q, k, v = (lang.reshape(b, lang.make_shape(b, 1, h, n, d), t) for t, h, n in ((q, H, S), (k, KV, T), (v, KV, T)))
        q, k, v = q + q - q, k + k - k, v + v - v
        a = lang.matmul(b, q, lang.transpose(b, 2, 3, helpers.repeat_kv(b, H // KV, k)))
        sh = lang.shape(b, a)
        a = a / lang.constant(b, float(np.sqrt(np.float32(d))), sh)
        if causal:
            a = a + lang.broadcast(b, helpers.causal_mask(b, lang.to_nat(b, S)), sh)
        return [lang.matmul(b, nn.softmax(b, a), helpers.repeat_kv(b, H // KV, v))]
    (got,) = vectors.run(hip_bf16, f, 1, q.reshape(-1), k.reshape(-1), v.reshape(-1))
    q, k, v = q.astype(np.float64), *(np.repeat(t.astype(np.float64), H // KV, axis=0) for t in (k, v))
    s = q @ k.transpose(0, 2, 1) / float(np.sqrt(np.float32(d)))
    if causal:
        s[:, np.triu(np.ones((S, S), bool), 1)] = -np.inf
    p = np.exp(s - s.max(-1, keepdims=True))
    exact = (p / p.sum(-1, keepdims=True)) @ v
    assert_f32_sums(exact, got, d + T, f"{S} queries over {T} keys")


# The routed experts of 9 to 63 tokens: rows and gated values in f32 beside the bf16 matrices, an expert with no pair, with
# few, with more than a tile of 20 holds; sizes that the tile kernel takes and (fewer than 12 tokens,
# F = 96 or 136) those that it does not
@pytest.mark.gpu
@pytest.mark.parametrize("S,k,E,H,F", [(9, 2, 5, 256, 192), (11, 4, 7, 128, 64), (12, 4, 60, 128, 64), (30, 3, 4, 320, 256), (63, 4, 7, 64, 136), (63, 1, 3, 1024, 448),
                                       (40, 8, 9, 128, 64), (21, 2, 6, 128, 96)])
def test_experts_of_a_short_prompt(hip_bf16, S, k, E, H, F):
    g = np.random.default_rng(S * 10 + k)
    x = g.standard_normal((S, H)).astype(np.float32)
    x[1] *= np.float32(1e-8)
    x[2] *= np.float32(1e8)
    wg, wu = (vectors.bf16_round((g.standard_normal((E, F, H)) * H ** -0.5).astype(np.float32)) for _ in range(2))
    wd = vectors.bf16_round((g.standard_normal((E, H, F)) * F ** -0.5).astype(np.float32))
    idx = g.choice(E - 1, (S, k), p=np.r_[0.7, np.full(E - 2, 0.3 / (E - 2))]).astype(np.uint32)    # the last expert has none

    def f(b, x, idx, wg, wu, wd):
        x = lang.reshape(b, lang.make_shape(b, S, 1, H), x)
        x = x + x - x
        out = []
        for i in range(k):
            slot = lang.get(b, 1, i, idx)
            sel = lambda w: lang.transpose(b, 1, 2, lang.index(b, 0, slot, w))      # noqa: B023
            out.append(lang.matmul(b, nn.silu(b, lang.matmul(b, x, sel(wg))) * lang.matmul(b, x, sel(wu)), sel(wd)))
        return out
    hip_bf16.launch_counts(reset=True)
    got = vectors.run(hip_bf16, f, k, x.reshape(-1), idx, wg, wu, wd)
    counts = hip_bf16.launch_counts(reset=True)
    assert (counts.get("gemm_experts_bf16", 0), counts.get("experts_route", 0)) == ((2, 1) if S >= 12 and H % 64 == F % 64 == 0 else (0, 0)), counts
    wg, wu, wd, x = (a.astype(np.float64) for a in (wg, wu, wd, x))
    for i in range(k):
        e = idx[:, i]
        gate, up = (np.einsum("sh,sfh->sf", x, w[e]) for w in (wg, wu))
        exact = np.einsum("sf,shf->sh", gate / (1 + np.exp(-np.maximum(gate, -700))) * up, wd[e])
        assert_f32_sums(exact, got[i], H + F, f"slot {i}")
