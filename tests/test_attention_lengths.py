"""One-pass attention (models/llama.rs:95-107, gemma3.rs:153-186) at numbers of queries and keys that are no multiple of
anything: mask rows and transposed values are padded for the 16-byte loads of the kernel, and a prompt of a few tokens
takes the same single launch (in bf16 mode from 9 tokens on: test_f32_operands.py has the rest)."""
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
        three = 128 < S < 512 or d == 256 if be is hip else S <= 8      # (two products and a softmax at these lengths)
        assert counts.get("attn_prefill", 0) == (0 if three else 1), counts
        check(ref, got, f"attention over {S} keys")


# every pair visible: steps without mask values (a maximum over raw scores, the scale in the exponent) beside the ragged last
# one; a scale that turns the order of the scores around, none at all, and scores that one key dominates
@pytest.mark.gpu
@pytest.mark.parametrize("H,KV,S,d", [(4, 2, 200, 64), (40, 8, 523, 64), (2, 1, 193, 128), (6, 3, 129, 256)])
@pytest.mark.parametrize("scale,loud", [(8.0, 1.0), (-6.0, 1.0), (None, 0.2), (8.0, 60.0)])
def test_attention_without_a_mask(oracle, hip_bf16, H, KV, S, d, scale, loud):
    g = np.random.default_rng(S + d)
    q, k, v = (vectors.bf16_round(g.standard_normal((1, h, S, d)).astype(np.float32)) for h in (H, KV, KV))
    q = vectors.bf16_round(q * np.float32(loud))

    def f(b, q, k, v):
        q, k, v = q + q - q, k + k - k, v + v - v
        attn = lang.matmul(b, q, lang.transpose(b, 2, 3, helpers.repeat_kv(b, H // KV, k)))
        if scale is not None:
            attn = attn / lang.constant(b, scale, lang.shape(b, attn))
        return lang.matmul(b, nn.softmax(b, attn), helpers.repeat_kv(b, H // KV, v))
    (ref,) = vectors.run(oracle, f, 1, q, k, v)
    (got,) = vectors.run(hip_bf16, f, 1, q, k, v)
    parity.assert_bf16(ref, got, f"{S} keys, scale {scale}")


@pytest.mark.gpu
@pytest.mark.parametrize("tokens", [67, 259])
def test_rotation_in_the_projections_launch_at_odd_lengths(oracle, hip_bf16, tokens):
    llama_tests.test_llama_prefill_rotates_in_the_projections_launch(oracle, hip_bf16, tokens, 8, 2, 2)


@pytest.mark.gpu
@pytest.mark.parametrize("batch,tokens,heads,kv_heads,head_dim", [(3, 67, 8, 8, 64), (2, 134, 4, 4, 128)])
def test_rotation_of_several_odd_sequences(oracle, hip_bf16, batch, tokens, heads, kv_heads, head_dim):
    """Four rows of a tile may belong to two sequences: the transposed values are stored one by one there."""
    moe_tests.test_qwen_prefill_biases_and_rotation_in_the_projections_launch(oracle, hip_bf16, batch, tokens, heads, kv_heads, head_dim)


# One query over long caches: kv heads shared by 2 to 8 query heads (the matrix-core form, from 881 keys or, heads of 128, from
# 40960 keys over all heads on) or none (the vector form at every length), last ranges that are short; the step's own rows go
# into the cache through the same launch.
@pytest.mark.gpu
@pytest.mark.parametrize("H,KV,d,T,steps", [(4, 1, 64, 881, 2), (8, 8, 128, 129, 3), (4, 2, 128, 515, 2), (16, 2, 64, 2049, 2),
                                            (2, 1, 128, 4100, 1), (4, 2, 64, 1300, 2), (16, 2, 128, 2559, 1), (2, 2, 64, 1000, 1)])
def test_decode_over_a_long_cache(oracle, hip, H, KV, d, T, steps):
    cfg = llm.Config(hidden_size=H * d, intermediate_size=64, num_hidden_layers=1, num_attention_heads=H, num_key_value_heads=KV,
                     vocab_size=97, rms_norm_eps=1e-5, rope_theta=10000.0)
    arrays = llm.random_init.llama_params(cfg, seed=T, std=0.08)
    g = np.random.default_rng(T)
    kv = [g.standard_normal((1, KV, T, d)).astype(np.float32) for _ in range(2)]
    runners = []
    for be in (oracle, hip):
        r = llm.CachedRunner(be, cfg, arrays, T + 8)
        # (rotations at small positions: an angle of hundreds of radians in f32 is itself off by T * 2^-24, which is the
        # tables' error on both sides and not this launch's)
        r.batch, r.pos, r.kv = 1, 3, [be.tensor(a) for a in kv]
        runners.append(r)
    hip.trace(2)
    for i, token in enumerate((5, 11, 90)[:steps + 1]):     # (the first step copies the cache, the following ones append)
        hip.trace_reset()
        hip.launch_counts(reset=True)
        out = [r.step(token)[1] for r in runners]
        parity.assert_f32(oracle.to_vec(out[0]), hip.to_vec(out[1]), f"token {token}")
        assert hip.launch_counts(reset=True).get("attn_decode") == 1
        keys = T + i + 1
        group = H > KV and (keys > 880 if d == 64 else H * keys >= 40960)
        names = [n for n in hip.trace_report() if n.startswith("attn_decode[")]
        assert len(names) == 1 and names[0].startswith("attn_decode[group," if group else "attn_decode[split,"), names
    hip.trace(0)
    for a, b in zip(runners[0].kv, runners[1].kv):
        parity.assert_f32(oracle.to_vec(a), hip.to_vec(b), "cache")


def leave_nan_in_memory(be, *sizes):
    """Blocks of these many bytes, filled with NaN and given back: the next allocations of their size classes get them."""
    be.sync()
    held = [be.tensor(np.full(n // 4, np.nan, np.float32)) for n in sizes for _ in range(4)]
    be.sync()
    del held


# What a cache's room to grow holds before it is written must not reach a result: an appending step of each decode kernel,
# whose last range of keys ends inside a tile (one workgroup; split keys; the matrix-core form, with one and two tiles of a
# pass past the end).
@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["f32", "bf16"])
@pytest.mark.parametrize("H,KV,d,T", [(4, 2, 64, 20), (4, 2, 64, 300), (4, 1, 64, 881), (16, 2, 64, 2049), (4, 2, 128, 129), (16, 4, 128, 2565)])
def test_unwritten_rows_of_a_cache_stay_out(oracle, hip, hip_bf16, mode, H, KV, d, T):
    be, check = (hip, parity.assert_f32) if mode == "f32" else (hip_bf16, parity.assert_bf16)
    cfg = llm.Config(hidden_size=H * d, intermediate_size=64, num_hidden_layers=1, num_attention_heads=H, num_key_value_heads=KV,
                     vocab_size=97, rms_norm_eps=1e-5, rope_theta=10000.0)
    arrays = llm.random_init.llama_params(cfg, seed=T, std=0.08)
    rounded = {k: (vectors.bf16_round(a) if a.ndim >= 2 else a) for k, a in arrays.items()}
    g = np.random.default_rng(T)
    kv = [vectors.bf16_round(g.standard_normal((1, KV, T, d)).astype(np.float32)) for _ in range(2)]
    room = 64
    while room < 2 * (T + 1):
        room *= 2
    ref, got = (llm.CachedRunner(b, cfg, rounded, T + 8) for b in (oracle, be))
    for r in (ref, got):
        # (uploaded as vectors: a cache is f32 in both modes)
        r.batch, r.pos, r.kv = 1, 3, [r.be.reshape(r.be.tensor(a.reshape(-1)), a.shape) for a in kv]
    leave_nan_in_memory(be, KV * room * d * 4)
    for token in (5, 11, 90):     # (the first step copies the cache, the following ones append)
        want, have = (r.be.to_vec(r.step(token)[1]) for r in (ref, got))
        assert np.isfinite(have).all(), f"token {token}"
        check(want, have, f"token {token}")


@pytest.mark.gpu
@pytest.mark.parametrize("H,KV,S,d", [(4, 2, 7, 64), (2, 2, 33, 128), (2, 1, 130, 64), (4, 1, 67, 256), (64, 64, 523, 64)])
def test_what_memory_held_stays_out_of_a_prompt(oracle, hip, hip_bf16, H, KV, S, d):
    """The padding of mask rows and transposed values is written, and rows past the last key never count."""
    g = np.random.default_rng(S + d)
    q, k, v = (vectors.bf16_round(g.standard_normal((1, h, S, d)).astype(np.float32)) for h in (H, KV, KV))
    f = attention(H, KV, S, d, 0)
    (ref,) = vectors.run(oracle, f, 1, q, k, v)
    for be, check in ((hip, parity.assert_f32), (hip_bf16, parity.assert_bf16)):
        leave_nan_in_memory(be, *(256 << i for i in range(13)), 1 << 20, 2 << 20)
        (got,) = vectors.run(be, f, 1, q, k, v)
        assert np.isfinite(got).all()
        check(ref, got, f"attention over {S} keys")


def attention_under(S, T, rep):
    def f(b, q, k, v, hidden):
        q, k, v = q + q - q, k + k - k, v + v - v
        attn = lang.matmul(b, q, lang.transpose(b, 2, 3, helpers.repeat_kv(b, rep, k)))
        sh = lang.shape(b, attn)
        mask = hidden * lang.constant(b, helpers.F32_MIN, lang.shape(b, hidden))
        attn = attn / lang.constant(b, 8.0, sh) + lang.broadcast(b, mask, sh)
        return lang.matmul(b, nn.softmax(b, attn), helpers.repeat_kv(b, rep, v))
    return f


def attention_in_numpy(q, k, v, hidden, rep):
    out = np.empty_like(q)      # (the oracle takes half a minute for the longest of these)
    for h in range(q.shape[1]):
        p = q[0, h] @ k[0, h // rep].T / np.float32(8) + hidden * np.float32(helpers.F32_MIN)
        p = np.exp(p - p.max(1, keepdims=True))
        out[0, h] = p @ v[0, h // rep] / p.sum(1, keepdims=True)
    return out


# Heads of 64 in two key groups of a query tile, 64 and 32 keys a step (by how many workgroups there are); heads of 128 and 256 as two
# halves of the values' dims, in two key groups of 32 or 64 queries, in one, and many heads of 128 undivided.  Key tiles seen by none, some or all of
# a query tile's rows at random (odd numbers of live steps, a group without any), rows that see no key at all, and more key tiles
# than the bit masks hold (T = 4100), heads that do not divide by the dies.
@pytest.mark.gpu
@pytest.mark.parametrize("H,KV,S,T,d", [(48, 6, 321, 321, 64), (65, 13, 257, 257, 64), (64, 8, 641, 641, 64), (322, 2, 65, 4100, 64),
                                         (16, 4, 200, 200, 128), (64, 8, 193, 193, 128), (80, 8, 200, 200, 128), (200, 8, 257, 257, 128),
                                         (4, 1, 200, 200, 256), (62, 2, 193, 193, 256), (80, 8, 131, 131, 256), (4, 4, 40, 33, 256)])
def test_parts_of_a_query_tile(hip_bf16, H, KV, S, T, d):
    g = np.random.default_rng(S + T)
    q = vectors.bf16_round(g.standard_normal((1, H, S, d)).astype(np.float32))
    k, v = (vectors.bf16_round(g.standard_normal((1, KV, T, d)).astype(np.float32)) for _ in range(2))
    tiles = g.integers(0, 3, ((S + 63) // 64, (T + 31) // 32))       # 0: hidden, 1: in part, 2: seen
    tiles[0] = 0
    tiles[0, (T - 1) // 32] = 2                                       # one live step for the first 64 queries
    per = np.repeat(np.repeat(tiles, 64, 0)[:S], 32, 1)[:, :T]
    hidden = np.where(per == 1, g.integers(0, 2, (S, T)), per == 0).astype(np.float32)
    hidden[[3, S - 1]] = 1
    f = attention_under(S, T, H // KV)
    ref = attention_in_numpy(q, k, v, hidden, H // KV)
    hip_bf16.launch_counts(reset=True)
    (got,) = vectors.run(hip_bf16, f, 1, q, k, v, hidden)
    assert hip_bf16.launch_counts(reset=True).get("attn_prefill") == 1
    parity.assert_bf16(ref, got, f"{S} queries of {T} keys")


# Heads of 64 whose keys are one step (test_kernel_choice.py asserts its kernel): full, ragged, of a length that is no multiple of four and of
# one that is; more queries than keys; pairs hidden at random, rows that see no key, a key that no row sees
@pytest.mark.gpu
@pytest.mark.parametrize("H,KV,S,T", [(4, 2, 37, 37), (8, 8, 64, 64), (2, 1, 200, 40), (6, 3, 17, 63), (4, 4, 33, 36), (32, 8, 9, 10)])
def test_keys_of_one_step(hip_bf16, H, KV, S, T):
    g = np.random.default_rng(S + T)
    q = vectors.bf16_round(g.standard_normal((1, H, S, 64)).astype(np.float32))
    k, v = (vectors.bf16_round(g.standard_normal((1, KV, T, 64)).astype(np.float32)) for _ in range(2))
    hidden = g.integers(0, 2, (S, T)).astype(np.float32)
    hidden[:, T - 2], hidden[:, 1] = 1, 0
    hidden[[3, S - 1]] = 1
    f = attention_under(S, T, H // KV)
    leave_nan_in_memory(hip_bf16, *(256 << i for i in range(13)), 1 << 20, 2 << 20)
    hip_bf16.launch_counts(reset=True)
    (got,) = vectors.run(hip_bf16, f, 1, q, k, v, hidden)
    counts = hip_bf16.launch_counts(reset=True)
    assert counts.get("attn_prefill") == 1 and "attn_mask_tiles" not in counts, counts
    parity.assert_bf16(attention_in_numpy(q, k, v, hidden, H // KV), got, f"{S} queries of {T} keys")


# Two views of one mask, alike but for their row stride: the first T columns of [S, 2 T] and the first S rows of the same values
# as [2 S, T].  What one of them hides from every query the other shows to half of them.
@pytest.mark.gpu
@pytest.mark.parametrize("S,T", [(64, 128), (200, 192), (64, 132)])
@pytest.mark.parametrize("order", [0, 1])
def test_views_of_one_mask(oracle, hip, hip_bf16, S, T, order):
    g = np.random.default_rng(S + T)
    qkv = [vectors.bf16_round(g.standard_normal((1, h, n, 64)).astype(np.float32)) for h, n in ((4, S), (2, T), (2, T)) * 2]
    mask = np.zeros((S, 2 * T), np.float32)
    mask[:, 64:T] = helpers.F32_MIN

    def f(b, *a):     # (the mask is uploaded as a vector: f32)
        views = [lang.slice(b, 1, 0, T, lang.reshape(b, lang.make_shape(b, S, 2 * T), a[6])),
                 lang.slice(b, 0, 0, S, lang.reshape(b, lang.make_shape(b, 2 * S, T), a[6]))]
        out = [None, None]
        for i in (order, 1 - order):
            q, k, v = (x + x - x for x in a[3 * i:3 * i + 3])
            attn = lang.matmul(b, q, lang.transpose(b, 2, 3, helpers.repeat_kv(b, 2, k)))
            sh = lang.shape(b, attn)
            attn = attn / lang.constant(b, 8.0, sh) + lang.broadcast(b, views[i], sh)
            out[i] = lang.matmul(b, nn.softmax(b, attn), helpers.repeat_kv(b, 2, v))
        return out if order == 0 else out[::-1]
    ref = vectors.run(oracle, f, 2, *qkv, mask.reshape(-1))
    for be, check in ((hip, parity.assert_f32), (hip_bf16, parity.assert_bf16)):
        be.launch_counts(reset=True)
        both = vectors.run(be, f, 2, *qkv, mask.reshape(-1))
        assert be.launch_counts(reset=True).get("attn_prefill", 0) == (0 if be is hip and T > 128 else 2)
        for r, got in zip(ref, both):
            check(r, got, "one view of the mask")
