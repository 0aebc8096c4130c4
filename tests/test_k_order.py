"""bf16 products of few rows whose weight rows lie a multiple of 4 KB apart, and the routed experts' products on such weights: column
tiles start at different k (KOrder), go to the end of their slice and then take what lies before.  Every kernel that does so, one tile
and many, slices, an odd number of k-steps, both forms of the stacked gate / up tile, values that would show a step taken twice.
test_kernel_choice.py holds the lists below to what they say: the kernel, the slices, and that the order is on or, in the lists of
the others, off."""
import numpy as np
import pytest

import test_large_tiles as large
import test_llama_parity as llama_tests
import vectors

lang, nn = vectors.cg.lang, vectors.cg.nn

# the direct-to-LDS kernel with k-groups, two stages, the scheduled loop, eight wavefronts; tiles of 128 x 256
GROUPS, STAGES, SCHEDULED, EIGHT = "dma_kernelILi64ELi64ELi2ELi2ELb%dELi8E", "dma_kernelILi64ELi64ELi2ELi2ELb%dELi2E", \
    "dma_kernelILi128ELi128ELi2ELi2ELb%dELi5E", "dma_kernelILi128ELi128ELi2ELi4ELb%dELi4E"
HALF = "ring_kernelILi%dELi1E"

# rows, columns, k, kernel, slices
PRODUCTS = [(17, 16384, 2048, GROUPS, 1), (64, 8200, 2048, GROUPS, 1), (64, 4096, 8192, GROUPS, 4), (17, 8000, 4096, GROUPS, 2), (64, 16500, 2048, STAGES, 1),
            (40, 33000, 4096, STAGES, 1), (128, 16400, 2048, SCHEDULED, 1), (128, 32000, 2048, SCHEDULED, 1), (128, 4100, 8192, SCHEDULED, 4), (100, 33000, 2048, HALF, 1)]
OTHER_PRODUCTS = [(17, 4100, 2048, GROUPS, 2), (65, 2100, 4096, EIGHT, 8), (129, 4100, 2048, EIGHT, 2)]    # slices of less than 2048 values; more rows

# ... and the values from one row of weights to the next, of which k are used: 33 and 49 k-steps, and 33 in each of four slices
PARTS_OF_ROWS = [(64, 9000, 2112, 4096, GROUPS, 1), (17, 16400, 2112, 4096, STAGES, 1), (128, 16400, 3136, 4096, SCHEDULED, 1), (100, 33000, 2112, 4096, HALF, 1),
                 (64, 2100, 8448, 10240, GROUPS, 4), (100, 4100, 8448, 10240, SCHEDULED, 4)]
OTHER_PARTS_OF_ROWS = [(17, 300, 2112, 4096, GROUPS, 8), (100, 2100, 3136, 4096, EIGHT, 4)]

SIGMOIDS = [(64, 8200, 2048, GROUPS), (100, 16400, 2048, EIGHT)]

# rows, hidden columns, k, kernel of the stacked product
GATED64, GATED128, GATED_WIDE = "dma_kernelILi64ELi64ELi2ELi1ELb1ELi8ELb1E", "dma_kernelILi128ELi64ELi4ELi1ELb1ELi5ELb1E", "dma_kernelILi128ELi128ELi4ELi2ELb1ELi4ELb1E"
GATED = [(17, 4160, 2048, GATED64), (64, 8200, 2048, GATED64), (65, 8192, 2048, GATED128), (128, 2048, 4096, GATED128), (100, 1040, 4096, GATED128),
         (100, 12000, 2048, GATED_WIDE), (100, 16640, 2048, HALF)]
OTHER_GATED = [(200, 2048, 2048, GATED128)]

# tokens, the kernel of both products, whether the order is on for the product with 2048 values of k
EXPERTS = [(20, "moe_gemm_dma_kernel", 1), (90, "moe_gemm_dma_kernel", 1), (330, "moe_ring_kernel", 1), (480, "moe_ring_kernel", 1), (700, "moe_ring_kernel", 0)]


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [c[:3] for c in PRODUCTS + OTHER_PRODUCTS])
def test_product(hip_bf16, M, N, K):
    large.test_product(hip_bf16, M, N, K)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(64, 8200, 2048), (64, 4096, 8192), (64, 16500, 2048), (128, 16400, 2048)])
def test_infinities(hip_bf16, M, N, K):
    large.test_infinities(hip_bf16, M, N, K)


# rows of weights of which a slice of columns is used, a view
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,apart", [c[:4] for c in PARTS_OF_ROWS + OTHER_PARTS_OF_ROWS])
def test_part_of_every_row(hip_bf16, M, N, K, apart):
    g = np.random.default_rng(K)
    x, w = large.draw(g, (1, M, K)), large.draw(g, (N, apart))

    def f(b, x, w):
        return [large.linear(b, x, lang.slice(b, 1, 64, K, w), N, K)]
    (got,) = vectors.run(hip_bf16, f, 1, x, w)
    ref, bound = large.product_and_bound(x[0], w[:, 64:64 + K])
    assert np.all(np.abs(got[0] - ref) <= bound)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [c[:3] for c in SIGMOIDS])
def test_sigmoid(hip_bf16, M, N, K):
    g = np.random.default_rng(N)
    x, w = large.draw(g, (1, M, K)), large.draw(g, (N, K), K ** -0.5)
    (got,) = vectors.run(hip_bf16, lambda b, x, w: [nn.sigmoid(b, large.linear(b, x, w, N, K))], 1, x, w)
    y, bound = large.product_and_bound(x[0], w)
    # a sigmoid's slope is 1/4 at most; its exponential, the sum and the quotient are rounded to f32
    assert np.all(np.abs(got[0] - 1 / (1 + np.exp(-y))) <= bound / 4 + 4 * 2.0 ** -24)


@pytest.mark.gpu
@pytest.mark.parametrize("act", ["silu", "gelu"])
@pytest.mark.parametrize("M,F,K", [c[:3] for c in GATED + OTHER_GATED])
def test_gated(hip_bf16, M, F, K, act):
    large.test_gated(hip_bf16, M, F, K, act)


# (q / k / v that rotate start at the same k)
@pytest.mark.gpu
@pytest.mark.parametrize("tokens", [17, 40, 128])
def test_rotated(oracle, hip_bf16, tokens):
    llama_tests.test_llama_prefill_rotates_in_the_projections_launch(oracle, hip_bf16, tokens, 32, 8, 1)


# two choices of five experts by few tokens (f32 rows as planes), by some and by many (tiles of 128 x 256), one expert crowded and one
# without tokens; gate and up of long rows, or down; too many tokens to an expert for the order to change
@pytest.mark.gpu
@pytest.mark.parametrize("S", [c[0] for c in EXPERTS])
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
