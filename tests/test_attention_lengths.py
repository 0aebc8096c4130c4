"""One-pass attention (models/llama.rs:95-107, gemma3.rs:153-186) at numbers of queries and keys that are no multiple of
anything: mask rows and transposed values are padded for the 16-byte loads of the kernel, and a prompt of a few tokens
takes the same single launch."""
import importlib

import numpy as np
import pytest

import parity
import test_llama_parity as llama_tests
import test_moe_gemma_parity as moe_tests
import vectors

lang, nn = vectors.cg.lang, vectors.cg.nn
llm = importlib.import_module("catgrad-rs_amd.llm")
helpers = llm.helpers


def attention(H, KV, S, d, window):
    model = llm.gemma3.Gemma3Model(llm.Config(), S)

    def f(b, q, k, v):
        q, k, v = q + q - q, k + k - k, v + v - v      # computed f32 values
        attn = lang.matmul(b, q, lang.transpose(b, 2, 3, helpers.repeat_kv(b, H // KV, k)))
        sh = lang.shape(b, attn)
        attn = attn / lang.constant(b, float(np.sqrt(np.float32(d))), sh)
        n = lang.to_nat(b, S)
        mask = model.window_mask(b, n, window) if window else helpers.causal_mask(b, n)
        attn = attn + lang.broadcast(b, mask, sh)
        return lang.matmul(b, nn.softmax(b, attn), helpers.repeat_kv(b, H // KV, v))
    return f


# the smallest, both sides of a 32-query / 64-key tile, of the 64- and 128-query tiles, each width of head
@pytest.mark.gpu
@pytest.mark.parametrize("H,KV,S,d,window", [(4, 2, 2, 64, 0), (4, 2, 7, 64, 0), (2, 2, 33, 64, 5), (8, 8, 65, 64, 0), (2, 1, 130, 64, 70),
                                             (4, 4, 37, 128, 0), (2, 1, 129, 128, 40), (4, 1, 31, 256, 0), (4, 1, 67, 256, 30),
                                             (64, 64, 523, 64, 0), (8, 2, 1027, 64, 0)])
def test_attention_of_any_length(oracle, hip, hip_bf16, H, KV, S, d, window):
    g = np.random.default_rng(S + d)
    # values bf16 storage keeps, so that the oracle and both modes work on the same numbers
    q, k, v = (vectors.bf16_round(g.standard_normal((2 if S < 500 else 1, h, S, d)).astype(np.float32)) for h in (H, KV, KV))
    f = attention(H, KV, S, d, window)
    (ref,) = vectors.run(oracle, f, 1, q, k, v)
    for be, check in ((hip, parity.assert_f32), (hip_bf16, parity.assert_bf16)):
        be.launch_counts(reset=True)
        (got,) = vectors.run(be, f, 1, q, k, v)
        counts = be.launch_counts(reset=True)
        three = be is hip and 128 < S < 512      # (f32: two products and a softmax at these lengths)
        assert sum(counts.get(n, 0) for n in ("attn_prefill", "attn_short", "attn_ragged")) == (0 if three else 1), counts
        check(ref, got, f"attention over {S} keys")


@pytest.mark.gpu
@pytest.mark.parametrize("tokens", [67, 259])
def test_rotation_in_the_projections_launch_at_odd_lengths(oracle, hip_bf16, tokens):
    llama_tests.test_llama_prefill_rotates_in_the_projections_launch(oracle, hip_bf16, tokens, 8, 2, 2)


@pytest.mark.gpu
@pytest.mark.parametrize("batch,tokens,heads,kv_heads,head_dim", [(3, 67, 8, 8, 64), (2, 134, 4, 4, 128)])
def test_rotation_of_several_odd_sequences(oracle, hip_bf16, batch, tokens, heads, kv_heads, head_dim):
    """Four rows of a tile may belong to two sequences: the transposed values are stored one by one there."""
    moe_tests.test_qwen_prefill_biases_and_rotation_in_the_projections_launch(oracle, hip_bf16, batch, tokens, heads, kv_heads, head_dim)
