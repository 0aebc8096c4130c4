"""bf16 products of few rows whose weight rows lie a multiple of 4 KB apart, and the routed experts' products on such weights: column
tiles start at different k (KOrder), go to the end of their slice and then take what lies before.  Every kernel that does so, one tile
and many, slices, an odd number of k-steps, both forms of the stacked gate / up tile, values that would show a step taken twice."""
import numpy as np
import pytest

import test_large_tiles as large
import test_llama_parity as llama_tests
import vectors

lang, nn = vectors.cg.lang, vectors.cg.nn


# 64 x 64 tiles with k-groups and, of more tiles than CUs, with two stages; 65 rows on; slices; less than a tile
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(17, 4100, 2048), (64, 16500, 2048), (40, 33000, 4096), (65, 2100, 4096), (128, 16400, 2048), (100, 2048, 8192),
                                   (33, 2048, 8192), (128, 32000, 2048), (17, 130, 6144), (129, 4100, 2048)])
def test_product(hip_bf16, M, N, K):
    large.test_product(hip_bf16, M, N, K)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(17, 4100, 2048), (100, 2048, 8192), (64, 16500, 2048)])
def test_infinities(hip_bf16, M, N, K):
    large.test_infinities(hip_bf16, M, N, K)


# rows 4096 values apart of which 33, 35 and 49 k-steps are used: slices of columns are views
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(17, 300, 2112), (64, 4100, 2240), (100, 2100, 3136)])
def test_part_of_every_row(hip_bf16, M, N, K):
    g = np.random.default_rng(K)
    x, w = large.draw(g, (1, M, K)), large.draw(g, (N, 4096))

    def f(b, x, w):
        return [large.linear(b, x, lang.slice(b, 1, 64, K, w), N, K)]
    (got,) = vectors.run(hip_bf16, f, 1, x, w)
    ref, bound = large.product_and_bound(x[0], w[:, 64:64 + K])
    assert np.all(np.abs(got[0] - ref) <= bound)


@pytest.mark.gpu
@pytest.mark.parametrize("act", ["silu", "gelu"])
@pytest.mark.parametrize("M,F,K", [(17, 4160, 2048), (64, 8200, 2048), (65, 8192, 2048), (128, 2048, 4096), (100, 1040, 4096), (200, 2048, 2048)])
def test_gated(hip_bf16, M, F, K, act):
    large.test_gated(hip_bf16, M, F, K, act)


@pytest.mark.gpu
@pytest.mark.parametrize("tokens", [17, 40, 128])
def test_rotated(oracle, hip_bf16, tokens):
    llama_tests.test_llama_prefill_rotates_in_the_projections_launch(oracle, hip_bf16, tokens, 32, 8, 1)


# two choices of five experts by few tokens (f32 rows as planes), by some and by many (tiles of 128 x 256), one expert crowded and one
# without tokens; gate and up of long rows, or down; too many tokens to an expert for the order to change
@pytest.mark.gpu
@pytest.mark.parametrize("S", [20, 90, 330, 700])
@pytest.mark.parametrize("F,H", [(192, 2048), (2048, 192)])
def test_experts(hip_bf16, S, F, H):
    E, k = 5, 2
    g = np.random.default_rng(S + F)
    x = large.draw(g, (S, 1, H))
    wg, wu = (large.draw(g, (E, F, H), H ** -0.5) for _ in range(2))
    wd = large.draw(g, (E, H, F), F ** -0.5)
    idx = np.stack([g.choice(np.array([0, 2, 3]), S, p=[.2, .7, .1]), np.full(S, 4)], 1).astype(np.uint32)

    def f(b, xv, iv, g_all, u_all, d_all):
        xv = xv + xv - xv
        total = None
        for i in range(k):
            slot = lang.get(b, 1, i, iv)
            sel = lambda w: lang.transpose(b, 1, 2, lang.index(b, 0, slot, w))
            y = lang.matmul(b, nn.silu(b, lang.matmul(b, xv, sel(g_all))) * lang.matmul(b, xv, sel(u_all)), sel(d_all))
            total = y if total is None else total + y
        return total
    hip_bf16.launch_counts(reset=True)
    (got,) = vectors.run(hip_bf16, f, 1, x, idx, wg, wu, wd)
    x64, ref, bound = x[:, 0].astype(np.float64), 0.0, 0.0
    for i in range(k):
        for e in range(E):
            rows = (idx[:, i] == e)[:, None]
            gate, up, d = x64 @ wg[e].T.astype(np.float64), x64 @ wu[e].T.astype(np.float64), wd[e].T.astype(np.float64)
            h = gate / (1 + np.exp(-gate)) * up
            # a gated value is rounded to bf16 (2^-8 of it at most, 2^-19 for exp2 and reciprocal) behind f32 sums of terms of size
            # K^-1/2 (as in test_large_tiles); then F additions
            dh = (2.0 ** -8 + 2.0 ** -19) * np.abs(h) + 4 * np.sqrt(H) * 2.0 ** -24 * (1.13 * np.abs(up) + np.abs(gate))
            ref = ref + rows * (h @ d)
            bound = bound + rows * ((dh + F * 2.0 ** -24 * np.abs(h)) @ np.abs(d))
    assert np.all(np.abs(got[:, 0] - ref) <= bound + 2.0 ** -23 * np.abs(ref))
