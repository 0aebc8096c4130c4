"""max(softmax(x)) and argmax(x) of the same rows in one pass (nn/mod.rs:162-171, ndarray.rs:455-480): rows of every length
and alignment, a wave / a workgroup / several workgroups to a row, and the values the folds treat specially."""
import numpy as np
import pytest

import vectors

lang, nn = vectors.cg.lang, vectors.cg.nn


def best(b, x):
    return lang.max(b, nn.softmax(b, x)), lang.argmax(b, x)


def run(be, x):
    if be.name.startswith("hip"):
        be.launch_counts(reset=True)
    out = vectors.run(be, best, 2, x)
    return out, (be.launch_counts(reset=True) if be.name.startswith("hip") else {})


# a few values; both sides of a wave's 1024; a piece of 8 or 16 and a bit; rows that start off a 16-byte boundary; few long
# rows (chunks) with a last chunk that is short
@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(1, 1), (3, 2), (5, 63), (7, 1024), (6, 1025), (300, 513), (2, 3, 4099), (257, 2049), (1, 8191),
                                   (1, 8192), (3, 20001), (1, 128256), (100, 8195)])
def test_best_of_rows(oracle, hip, hip_bf16, shape):
    g = np.random.default_rng(shape[-1])
    x = vectors.bf16_round((g.standard_normal(shape) * 3).astype(np.float32))     # (bf16 values: ties at the top are common)
    (p, a), _ = run(oracle, x)
    for be in (hip, hip_bf16):
        (gp, ga), counts = run(be, x)
        assert counts.get("softmax_best") == 1 and not any(n.startswith(("reduce", "row_fused")) for n in counts), counts
        # one f32 exponential and a sum of n of them on both sides: 1e-5
        assert np.allclose(gp, p, rtol=1e-5, atol=0) and np.array_equal(ga, a)


@pytest.mark.gpu
def test_best_of_rows_with_special_values(oracle, hip):
    x = np.random.default_rng(3).standard_normal((9, 70)).astype(np.float32)
    x[0, 5] = np.inf
    x[1, 69] = np.nan
    x[2] = -np.inf
    x[3, :69] = -np.inf
    x[4] = np.nan
    x[5] = 2.5
    x[6, 3], x[6, 66] = 90.0, -3e38
    x[7] = np.finfo(np.float32).min
    (p, a), _ = run(oracle, x)
    (gp, ga), _ = run(hip, x)
    assert np.allclose(gp, p, rtol=1e-5, atol=0, equal_nan=True) and np.array_equal(ga, a), (p, gp, a, ga)


# the same in rows of several groups of values to a thread, where the column is looked for in the group the largest was met in: equal
# largest values in different groups, waves and pieces, zeros of both signs, NaN of both signs beside and behind the largest
@pytest.mark.gpu
@pytest.mark.parametrize("n", [70, 1000, 1030, 4097, 9001, 40000])
def test_special_values_in_several_groups(oracle, hip, n):
    g = np.random.default_rng(n)
    x = vectors.bf16_round(-np.abs(g.standard_normal((14, n))).astype(np.float32))
    x[0, [0, n // 2, n - 1]] = 3.0                                         # the last of equal values
    x[1, [1, n // 3]] = 3.0
    x[2, [n // 4, n - 2]], x[2, n // 2] = 0.0, -0.0                         # +0 is the larger
    x[3, n // 2] = -0.0
    x[4] = np.where(np.arange(n) % 2, 0.0, -0.0)
    x[5, n // 2] = np.nan
    x[6, n // 3], x[6, n - 1] = np.float32(-np.nan), 5.0                    # (a NaN with its sign set is below everything)
    x[7, n - 1], x[7, 0] = np.nan, np.inf
    x[8, [3, n // 2]] = np.inf
    x[9] = -np.inf
    x[9, n // 2] = np.finfo(np.float32).min
    x[10] = np.float32(-np.nan)
    x[11, n // 2:] = -np.inf
    x[12] = np.nan
    (p, a), _ = run(oracle, x)
    (gp, ga), _ = run(hip, x)
    for r in range(len(x)):
        assert np.allclose(gp[r], p[r], rtol=1e-5, atol=0, equal_nan=True) and np.array_equal(ga[r], a[r]), (r, p[r], gp[r], a[r], ga[r])


# a wave to rows of more than 1024 values where there are many of them: 32 and 64 values to a thread
@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(1030, 1031), (1024, 2048), (2050, 2049), (2048, 4096), (2051, 4095), (2048, 4097)])
def test_a_wave_to_a_longer_row(oracle, hip, hip_bf16, shape):
    test_best_of_rows(oracle, hip, hip_bf16, shape)


# turns that end inside the row: exactly one, several, one and a part, of a wave and of a workgroup
@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(40, 1024), (1024, 1024), (2100, 2048), (9, 4096), (5, 12288), (7, 12289), (3, 4103), (2, 65536)])
def test_whole_turns(oracle, hip, hip_bf16, shape):
    test_best_of_rows(oracle, hip, hip_bf16, shape)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1024, 4096, 8192, 8200])
def test_special_values_in_whole_turns(oracle, hip, n):
    test_special_values_in_several_groups(oracle, hip, n)


# rows whose sum lies in many equal terms, which are all off to the same side: the largest value in front of every thread's others, or four
# distinct values.  Against 64 bits a term with d = x - max is off by 2^-23 for exp2, 2^-23 |d| for the rounded difference and product and
# 1.4e-8 |d| for log2 e; a sum goes through at most 16 additions to a partial sum of a group, two, one for each group that a thread meets
# (4096 values of a row), and 16 between threads and workgroups, with four more exponentials
@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["hip", "hip_bf16"])
@pytest.mark.parametrize("rows,n", [(64, 300), (64, 1024), (1024, 2000), (2048, 4000), (64, 4096), (256, 20000), (300, 131072), (3, 128256)])
def test_error_on_rows_of_few_values(request, mode, rows, n):
    be, g = request.getfixturevalue(mode), np.random.default_rng(n)
    below = np.linspace(0.25, 14, rows).astype(np.float32)[:, None]
    behind = np.repeat(-below, n, axis=1)
    behind[:, :min(n, 1024):4] = 0
    for x in (behind, -below * g.integers(0, 4, (rows, n)).astype(np.float32) / 3):
        x = vectors.bf16_round(x)
        (p, _), counts = run(be, x)
        assert counts.get("softmax_best") == 1, counts
        d = x.astype(np.float64)
        d -= d.max(axis=1, keepdims=True)
        e = np.exp(d)
        terms = (e * (2.0 ** -23 + np.abs(d) * (2.0 ** -23 + 1.4e-8))).sum(axis=1) / e.sum(axis=1)
        assert np.all(np.abs(p.ravel() * e.sum(axis=1) - 1) <= terms + (34 + n / 4096) * 2.0 ** -24 + 4 * 2.0 ** -23)


# what the two leave in memory is read back together where the rows are few: in either order, through a view, with more results held than
# there are buffers, again after their storage has served others, and by itself once cg_argmax_into has written it
@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 63, 64, 4096, 8192, 8193])
def test_results_read_one_after_the_other(hip, rows):
    cg = vectors.cg
    it, term = cg.Interpreter(hip, cg.stdlib()), vectors.Fn("best", 1, 2, best).term()
    g = np.random.default_rng(rows)
    xs = [g.standard_normal((rows, 8)).astype(np.float32) for _ in range(18 if rows == 63 else 3)]

    def check(out, x, order):
        e = np.exp(x.astype(np.float64) - x.max(1, keepdims=True))
        for i in order:
            got = hip.to_vec(out[i])
            assert np.array_equal(got, x.argmax(1)) if i else np.allclose(got, 1 / e.sum(1), rtol=1e-5, atol=0)
    for again in range(2):
        held = [it.run(term, [hip.tensor(x)]) for x in xs]
        for j, (out, x) in enumerate(zip(held, xs)):
            hip.realize(out[0])     # (asked for first, the column is found by itself)
            check(out, x, ((0, 1), (1, 0), (1, 1, 0, 0))[j % 3])
        del out
    seen = hip.reshape(held[0][1], (rows,))
    assert np.array_equal(hip.to_vec(seen), xs[0].argmax(1))
    other = hip.realize(hip.tensor(xs[1]))
    hip.argmax_into(other, held[0][1])
    assert np.array_equal(hip.to_vec(held[0][1]), xs[1].argmax(1)) and np.array_equal(hip.to_vec(seen), xs[1].argmax(1))
    check(held[0], xs[0], (0,))
    hip.argmax_into(hip.realize(hip.tensor(xs[2])), held[0][1])
    assert np.array_equal(hip.to_vec(held[0][1]), xs[2].argmax(1))


# an error that a kernel flags between the two reads is reported by the second, as if it crossed the bus by itself; the next ones are clean
@pytest.mark.gpu
@pytest.mark.parametrize("first", [0, 1])
def test_an_error_between_two_reads(hip, first):
    cg = vectors.cg
    x = np.random.default_rng(5).standard_normal((70, 9)).astype(np.float32)
    out = cg.Interpreter(hip, cg.stdlib()).run(vectors.Fn("best", 1, 2, best).term(), [hip.tensor(x)])
    a, zero = hip.realize(hip.tensor(np.arange(4, dtype=np.uint32))), hip.realize(hip.tensor(np.zeros(4, np.uint32)))
    hip.to_vec(out[first])
    hip.realize(hip.div(a, zero))
    with pytest.raises(cg.BackendPanic, match="divide by zero"):
        hip.to_vec(out[1 - first])
    assert np.array_equal(hip.to_vec(out[1]), x.argmax(1)) and hip.to_vec(out[0]).shape == (70,)
    hip.sync()
