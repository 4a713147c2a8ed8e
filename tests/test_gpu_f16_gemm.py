"""The any-shape fp16 matmul and the launches that take an operator's consumer along."""
import numpy as np
import pytest

from attention_superoptimizer_amd import graph as G
from helpers import assert_f16_close, normal_f16
from oracle import evaluate as orc
from test_gpu_f16 import _abi_matmul

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,m,n,k", [
    (1, 1, 8, 8),        # one chunk of everything
    (2, 5, 9, 63),       # no whole stage: the partial one alone
    (1, 17, 65, 65),     # one element past a tile, a stage and a chunk
    (3, 15, 71, 128),    # whole stages only, ragged columns
    (1, 3, 333, 3001),   # few tiles, long odd k: ranges of k, summed by the second launch
    (4, 65, 191, 257),
    (1, 300, 1001, 515),
    (1, 1000, 4001, 75),  # the largest tiles
    (2, 9, 7, 40),       # rows shorter than a chunk: element by element
])
def test_matmul_of_any_shape(rt, abi, batch, m, n, k):
    for a_cm, b_cm in ((0, 1), (0, 0), (1, 1), (1, 0)):
        a, b, got = _abi_matmul(rt, abi, batch, m, n, k, a_cm, b_cm, 5)
        assert_f16_close(got, orc.f16_matmul(a, b), what=f"[{batch},{m},{k}] . [{batch},{k},{n}], A cm {a_cm}, B cm {b_cm}")


def _execute(build, inputs, whole):
    """Every tensor of a graph after one run: of the whole graph at once, or operator by operator."""
    g = G.KNGraph()
    try:
        tensors = build(g)
        for t, a in zip(tensors, inputs):
            t.write_data(a)
        if whole:
            g.execute_all()
        else:
            for i in range(g.num_operators):
                g.execute(i)
        return [t.read_data() for t in tensors]
    finally:
        g.close()


@pytest.mark.parametrize("b,m,n,k", [(1, 1, 8, 16), (2, 33, 77, 65), (1, 40, 130, 3001), (1, 3, 6, 20), (1, 3600, 3700, 256),
                                     (1, 4090, 4096, 128)])
@pytest.mark.parametrize("op", ["exp", "silu", "add", "mul", "div", "rdiv"])
def test_consumer_in_the_matmul(rt, abi, op, b, m, n, k):
    def build(g):
        A, B, X = g.new_input((b, m, k)), g.new_input((b, k, n), layout="DmemColumnMajor"), g.new_input((b, m, n))
        C = g.matmul(A, B)
        E = g._unary(op, C) if op in ("exp", "silu") else g.div(X, C) if op == "rdiv" else g._binary(op, C, X)
        return A, B, X, C, E

    ins = [normal_f16([b, m, k], 0.2, 1), normal_f16([b, k, n], 0.2, 2), np.abs(normal_f16([b, m, n], 1.0, 3)) + np.float16(0.5)]
    for whole, single in zip(_execute(build, ins, True), _execute(build, ins, False)):
        np.testing.assert_array_equal(whole, single)


@pytest.mark.parametrize("b,m,n", [(1, 1, 1), (2, 3, 7), (1, 5, 2047), (1, 5, 4097), (2, 600, 513), (1, 1024, 65), (1, 1025, 4096), (1, 2, 20001)])
def test_softmax_rows(rt, abi, b, m, n):
    def build(g):
        X = g.new_input((b, m, n))
        E = g.exp(X)
        R = g.reduction(E, 2)
        return X, E, R, g.div(E, R)

    ins = [normal_f16([b, m, n], 0.5, 4)]
    whole, single = _execute(build, ins, True), _execute(build, ins, False)
    np.testing.assert_array_equal(whole[1], single[1])
    for w, s in zip(whole[2:], single[2:]):  # (another order of the row sum)
        assert_f16_close(w, s, rtol=2e-3, atol=1e-6, what="row sum or quotient")


def _odd_numbers(a, seed):
    """A few infinities and NaN at the edges and inside, and values whose products overflow fp16."""
    rng = np.random.default_rng(seed)
    a = a.copy()
    flat = a.reshape(-1)
    flat[-1], flat[0] = np.inf, -np.inf
    flat[rng.integers(0, flat.size, 3)] = np.nan
    flat[rng.integers(0, flat.size, 3)] = 60000
    return a


@pytest.mark.parametrize("batch,m,n,k", [
    (2, 33, 77, 65), (1, 3, 333, 3001), (1, 130, 200, 320), (2, 100, 136, 96), (1, 17, 4096, 512), (1, 2100, 4100, 64)])
def test_infinities_and_nan_stay_where_they_belong(rt, abi, monkeypatch, batch, m, n, k):
    """An infinity or NaN reaches the products it is part of and no other: padding of tiles, repeated rows and
    shifted chunks of k multiply nothing with it."""
    import test_gpu_f16
    monkeypatch.setattr(test_gpu_f16, "normal_f16", lambda d, std, seed: _odd_numbers(normal_f16(d, std, seed), seed))
    for a_cm, b_cm in ((0, 1), (0, 0), (1, 1), (1, 0)):
        a, b, got = _abi_matmul(rt, abi, batch, m, n, k, a_cm, b_cm, 5)
        with np.errstate(all="ignore"):
            want = np.matmul(a.astype(np.float32), b.astype(np.float32)).astype(np.float16)
        what = f"A cm {a_cm}, B cm {b_cm}"
        assert np.array_equal(np.isnan(got), np.isnan(want)), what
        assert np.array_equal(np.isposinf(got), np.isposinf(want)) and np.array_equal(np.isneginf(got), np.isneginf(want)), what
        ok = np.isfinite(want)
        assert ok.any()
        assert_f16_close(got[ok], want[ok], what=what)


@pytest.mark.parametrize("b,m,n,k", [(2, 33, 77, 65), (1, 40, 136, 320), (1, 16, 512, 512), (1, 40, 130, 3001)])
@pytest.mark.parametrize("op", ["exp", "silu", "add", "mul", "div", "rdiv"])
def test_consumer_of_numbers_out_of_range(rt, abi, op, b, m, n, k):
    def build(g):
        A, B, X = g.new_input((b, m, k)), g.new_input((b, k, n), layout="DmemColumnMajor"), g.new_input((b, m, n))
        C = g.matmul(A, B)
        return A, B, X, C, g._unary(op, C) if op in ("exp", "silu") else g.div(X, C) if op == "rdiv" else g._binary(op, C, X)

    ins = [_odd_numbers(normal_f16([b, m, k], 1.0, 1), 1), _odd_numbers(normal_f16([b, k, n], 1.0, 2), 2),
           _odd_numbers(normal_f16([b, m, n], 1.0, 3), 3)]
    ins[0][:, 0] = 0   # (a row of zeros: x / 0 and 0 / 0)
    ins[2][:, 0, ::2] = 0
    for whole, single in zip(_execute(build, ins, True), _execute(build, ins, False)):
        np.testing.assert_array_equal(whole, single)


@pytest.mark.parametrize("m,n", [(1, 7), (600, 513), (1024, 65), (1030, 4096), (5, 4097), (2, 20001)])
def test_softmax_rows_out_of_range(rt, abi, m, n):
    """Rows of -inf, rows with +inf or NaN, rows whose exponentials or whose sum overflow, rows that vanish."""
    def build(g):
        X = g.new_input((1, m, n))
        E = g.exp(X)
        R = g.reduction(E, 2)
        return X, E, R, g.div(E, R)

    x = normal_f16([1, m, n], 0.5, 4)
    kinds = [lambda r: r.fill(-np.inf), lambda r: r.__setitem__(n // 2, np.inf), lambda r: r.__setitem__(n - 1, np.nan),
             lambda r: r.__setitem__(0, 12), lambda r: r.fill(11), lambda r: r.fill(-20), lambda r: r.__setitem__(0, -np.inf)]
    for i in range(m):
        if m <= 5 or i % 3 == 0:
            kinds[(i + n) % len(kinds)](x[0, i])
    whole, single = _execute(build, [x], True), _execute(build, [x], False)
    np.testing.assert_array_equal(whole[1], single[1])
    for w, s in zip(whole[2:], single[2:]):
        assert np.array_equal(np.isnan(w), np.isnan(s)) and np.array_equal(np.isinf(w), np.isinf(s))
        ok = np.isfinite(s)
        # (one order of the fp32 row sum against another: two fp16 places, where they are normal numbers)
        assert_f16_close(w[ok], s[ok], rtol=2e-3, atol=1e-6, what="row sum or quotient")


@pytest.mark.parametrize("m,n,k", [
    (40, 2105, 1087), (126, 2105, 1151), (182, 1807, 1027), (300, 1027, 1343),  # 16, 17 and 20 stages and a part of one
    (126, 1300, 2049), (300, 2049, 1280), (603, 1220, 1408)])                   # 32; 20 and 22 whole stages
def test_matmul_of_many_stages(rt, abi, m, n, k):
    """Ranges long enough to be loaded four stages ahead: every remainder of their number by four, with and
    without a partial stage."""
    for a_cm, b_cm in ((0, 1), (0, 0), (1, 1)):
        a, b, got = _abi_matmul(rt, abi, 1, m, n, k, a_cm, b_cm, 5)
        assert_f16_close(got, orc.f16_matmul(a, b), what=f"[{m},{k}] . [{k},{n}], A cm {a_cm}, B cm {b_cm}")
