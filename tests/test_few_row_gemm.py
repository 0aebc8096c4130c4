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
