"""An expert that every token passes through beside the routed ones of a prefill, bf16 mode: tiles of the same two launches
(MoeGemmDesc::dense).  Row and column tiles that are partly filled, a dense expert whose down_proj is longer, as long and shorter than
the routed ones' - its tiles first, or spread among the others -, crowded and empty experts, either activation, and experts that do not join."""
import numpy as np
import pytest

import test_large_tiles as large
import vectors

lang, nn = vectors.cg.lang, vectors.cg.nn

# tokens, routed columns, width, dense columns, whether one launch takes both (8 columns' worth of routed tiles for the row tiles; k % 64)
CASES = [(300, 768, 1280, 320, True), (300, 768, 1280, 768, True), (257, 1024, 1280, 2176, True), (700, 1408, 1536, 1088, True),
         (128, 512, 2112, 192, True), (300, 768, 256, 320, False), (300, 768, 1280, 1000, False)]


def layer(act, k, F, H, FS):
    gate = nn.silu if act == "silu" else nn.gelu

    def f(b, xv, iv, g_all, u_all, d_all, sg, su, sd):
        xv = xv + xv - xv
        rows, total = lang.transpose(b, 0, 1, xv), None
        for i in range(k):
            slot = lang.get(b, 1, i, iv)
            sel = lambda w: lang.transpose(b, 1, 2, lang.index(b, 0, slot, w))
            y = lang.matmul(b, gate(b, lang.matmul(b, rows, sel(g_all))) * lang.matmul(b, rows, sel(u_all)), sel(d_all))
            total = y if total is None else total + y
        y = gate(b, large.linear(b, xv, sg, FS, H)) * large.linear(b, xv, su, FS, H)
        return [total, large.linear(b, y, sd, H, FS)]
    return f


@pytest.mark.gpu
@pytest.mark.parametrize("S,F,H,FS,joined", CASES)
@pytest.mark.parametrize("act", ["silu", "gelu"])
def test_dense_expert(hip_bf16, S, F, H, FS, joined, act):
    E, k = 5, 2
    g = np.random.default_rng(S + FS)
    x = large.draw(g, (1, S, H))
    wg, wu, sg, su = (large.draw(g, s, H ** -0.5) for s in ((E, F, H), (E, F, H), (FS, H), (FS, H)))
    wd, sd = large.draw(g, (E, H, F), F ** -0.5), large.draw(g, (H, FS), FS ** -0.5)
    idx = np.stack([g.choice(np.array([0, 2, 3]), S, p=[.2, .7, .1]), np.full(S, 4)], 1).astype(np.uint32)
    f = layer(act, k, F, H, FS)
    hip_bf16.launch_counts(reset=True)
    routed, dense = vectors.run(hip_bf16, f, 2, x, idx, wg, wu, wd, sg, su, sd)
    counts = hip_bf16.launch_counts()
    alone = {n: c for n, c in counts.items() if n.startswith("gemm") and n != "gemm_experts_bf16"}
    assert counts["gemm_experts_bf16"] == 2 and bool(alone) != joined, counts
    x64 = x[0].astype(np.float64)

    def expert(wg, wu, wd):  # the result, and what it may be off by (test_k_order.py has the terms)
        a, u, d = x64 @ wg.T.astype(np.float64), x64 @ wu.T.astype(np.float64), wd.T.astype(np.float64)
        if act == "silu":
            h = a / (1 + np.exp(-a)) * u
        else:
            h = 0.5 * a * (1 + np.tanh(0.7978845608028654 * (a + 0.044715 * a ** 3))) * u
        dh = (2.0 ** -8 + 2.0 ** -18) * np.abs(h) + 4 * np.sqrt(H) * 2.0 ** -24 * (1.13 * np.abs(u) + np.abs(a))
        return h @ d, (dh + wd.shape[1] * 2.0 ** -24 * np.abs(h)) @ np.abs(d)
    ref, bound = expert(sg, su, sd)
    assert np.all(np.abs(dense[0] - ref) <= bound)
    ref = bound = 0.0
    for e in range(E):
        y, dy = expert(wg[e], wu[e], wd[e])
        times = (idx == e).sum(1)[:, None]
        ref, bound = ref + times * y, bound + times * dy
    assert np.all(np.abs(routed[:, 0] - ref) <= bound + 2.0 ** -23 * np.abs(ref))


# Experts of several row tiles: which of them a pair lies in follows from the order in which the sort's atomics land, and from the other tokens.
# A routed row's sums come in the same order wherever it lies: the same bits in every run, and for the same tokens in another order.
@pytest.mark.gpu
@pytest.mark.parametrize("S,F,H,FS", [c[:4] for c in CASES[:4]] + [(2100, 512, 1024, 256)])
def test_the_same_bits_wherever_a_pair_lies(hip_bf16, S, F, H, FS):
    E, k = 5, 2
    g = np.random.default_rng(S + F)
    x = large.draw(g, (1, S, H))
    weights = [large.draw(g, s, s[-1] ** -0.5) for s in ((E, F, H), (E, F, H), (E, H, F), (FS, H), (FS, H), (H, FS))]
    idx = np.stack([g.choice(np.array([0, 2, 3]), S, p=[.2, .7, .1]), np.full(S, 4)], 1).astype(np.uint32)
    run = lambda order: vectors.run(hip_bf16, layer("silu", k, F, H, FS), 2, x[:, order], idx[order], *weights)
    routed, dense = run(np.arange(S))
    for again in range(4):
        r, d = run(np.arange(S))
        assert np.array_equal(r, routed) and np.array_equal(d, dense), again
        order = g.permutation(S)
        assert np.array_equal(run(order)[0], routed[order]), again


# The dense expert's down_proj on operands that are known exactly: gates of 64 (whose silu is 64 to the last bit) and up projections that pick
# a value of the token.  A sum of random terms in chains of n additions is off by 0.42 2^-24 sqrt(n / 2) - a rounding is 0.42 2^-24 of the
# partial sum, whose square grows evenly -, and an MFMA makes two additions for 16 values: 3.3e-7 for 5632 values in two chains, which is what
# they were in two slices, 4.7e-7 in one.
@pytest.mark.gpu
@pytest.mark.parametrize("S,FS", [(300, 5632), (300, 5696), (131, 2816)])
def test_the_sums_of_a_deep_down_projection(hip_bf16, S, FS):
    E, k, F, H = 5, 2, 768, 2048
    g = np.random.default_rng(FS)
    x = large.draw(g, (1, S, H))
    x[..., 0] = 1
    idx = np.stack([g.choice(np.array([0, 2, 3]), S), np.full(S, 4)], 1).astype(np.uint32)
    routed = [large.draw(g, s, s[-1] ** -0.5) for s in ((E, F, H), (E, F, H), (E, H, F))]
    sg, su, pick = np.zeros((FS, H), np.float32), np.zeros((FS, H), np.float32), g.integers(1, H, FS)
    sg[:, 0], su[np.arange(FS), pick] = 64, 1
    sd = large.draw(g, (H, FS), FS ** -0.5)
    hip_bf16.launch_counts(reset=True)
    _, dense = vectors.run(hip_bf16, layer("silu", k, F, H, FS), 2, x, idx, *routed, sg, su, sd)
    counts = hip_bf16.launch_counts()
    assert counts["gemm_experts_bf16"] == 2 and "gemm" not in counts, counts
    ref = 64 * x[0][:, pick].astype(np.float64) @ sd.T.astype(np.float64)
    off = np.linalg.norm(dense[0] - ref) / np.linalg.norm(ref)
    assert off <= 1.15 * 0.42 * 2.0 ** -24 * np.sqrt(FS / 16 / 2), off
