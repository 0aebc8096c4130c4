"""bf16 products of 17 to 128 rows (a short prompt): narrow tiles with k-groups, the stacked gate / up tile at each of its
widths, products split along k, and the rotating q/k/v launch on tiles of 64 rows."""
import importlib

import numpy as np
import pytest

import parity
import test_llama_parity as llama_tests
import test_moe_gemma_parity as moe_tests
import vectors

lang, nn = vectors.cg.lang, vectors.cg.nn


def gated_mlp(b, x, wg, wu, wd):
    def linear(x, w):      # [1, rows, in] by [out, in], as stdlib's linear does it
        n, k = w_shape[id(w)]
        return lang.matmul(b, x, lang.reshape(b, lang.make_shape(b, 1, k, n), lang.transpose(b, 0, 1, w)))
    w_shape = {id(wg): gated_mlp.up, id(wu): gated_mlp.up, id(wd): gated_mlp.down}
    x = x + x - x
    return [linear(nn.silu(b, linear(x, wg)) * linear(x, wu), wd)]


# rows on both sides of every tile height; columns that end inside a tile; k of one step and of many, deep enough to split
@pytest.mark.gpu
@pytest.mark.parametrize("rows", [17, 32, 33, 64, 65, 127, 128, 129, 200])
@pytest.mark.parametrize("K,F,N", [(64, 192, 64), (512, 1096, 200), (1152, 256, 2048), (256, 4160, 136)])
def test_gated_mlp_of_few_rows(oracle, hip_bf16, rows, K, F, N):
    g = np.random.default_rng(rows + K)
    x, wg, wu, wd = (vectors.bf16_round((g.standard_normal(s) * std).astype(np.float32))
                     for s, std in (((1, rows, K), 1.0), ((F, K), K ** -0.5), ((F, K), K ** -0.5), ((N, F), F ** -0.5)))
    gated_mlp.up, gated_mlp.down = (F, K), (N, F)
    (ref,) = vectors.run(oracle, gated_mlp, 1, x, wg, wu, wd)
    hip_bf16.launch_counts(reset=True)
    (got,) = vectors.run(hip_bf16, gated_mlp, 1, x, wg, wu, wd)
    counts = hip_bf16.launch_counts(reset=True)
    assert counts.get("gemm") == 2 and "swiglu_fused" not in counts, counts
    parity.assert_bf16(ref, got, f"{rows} rows")


@pytest.mark.gpu
@pytest.mark.parametrize("tokens", [17, 40, 64, 99, 128])
def test_rotation_in_the_projections_launch_of_few_rows(oracle, hip_bf16, tokens):
    llama_tests.test_llama_prefill_rotates_in_the_projections_launch(oracle, hip_bf16, tokens, 8, 2, 2)


@pytest.mark.gpu
@pytest.mark.parametrize("batch,tokens,heads", [(1, 40, 4), (3, 20, 4), (3, 41, 4), (1, 128, 4), (1, 101, 16)])
def test_rotation_of_wide_heads_of_few_rows(oracle, hip_bf16, batch, tokens, heads):
    moe_tests.test_qwen_prefill_biases_and_rotation_in_the_projections_launch(oracle, hip_bf16, batch, tokens, heads, heads, 128)


# more 64 x 64 tiles than the device has CUs: the form with two stages - one k-step, an odd number, many -, rows and columns
# that end inside a tile; and on both sides of the depth from which a product of few tiles is split along k
@pytest.mark.gpu
@pytest.mark.parametrize("batch,rows,K,N", [(130, 17, 64, 130), (300, 64, 128, 64), (5, 33, 192, 4001), (1, 40, 320, 16500), (90, 63, 704, 200),
                                            (1, 17, 960, 64), (1, 64, 1024, 64), (3, 40, 512, 136)])
def test_many_small_products(hip_bf16, batch, rows, K, N):
    g = np.random.default_rng(batch + rows)
    x, w = (vectors.bf16_round(g.standard_normal(s).astype(np.float32)) for s in ((batch, rows, K), (batch, N, K)))

    def f(b, x, w):
        return [lang.matmul(b, x, lang.transpose(b, 1, 2, w))]
    (got,) = vectors.run(hip_bf16, f, 1, x, w)
    exact = x.astype(np.float64) @ w.astype(np.float64).transpose(0, 2, 1)
    # (the operands are bf16 already: sums of K exact products in f32)
    err = np.linalg.norm(got - exact, axis=-1) / np.linalg.norm(exact, axis=-1)
    assert err.max() <= 4 * np.sqrt(K) * 2.0 ** -24, err.max()
