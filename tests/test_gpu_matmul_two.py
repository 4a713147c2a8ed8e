"""Two kernel-level matmuls of one input, with the element-wise operators that consume them, when a graph runs as a
whole (KNGraph.execute_all): the products against the fp64 oracle, what consumes them bit for bit against the same
operators run one by one on those products."""
import ctypes

import numpy as np
import pytest

from attention_superoptimizer_amd import _native as N
from attention_superoptimizer_amd import graph as G
from helpers import assert_f16_close, normal_f16
from oracle import evaluate as orc

pytestmark = pytest.mark.gpu
ROW, COL = "DmemRowMajor", "DmemColumnMajor"


class MatmulOut(ctypes.Structure):  # mi355_matmul_out
    _fields_ = [("B", ctypes.c_void_p), ("C", ctypes.c_void_p), ("op", ctypes.c_int), ("x_first", ctypes.c_int),
                ("X", ctypes.c_void_p), ("E", ctypes.c_void_p)]


def _taken(A, B, B2, X, C, E, C2, E2, form, b, m, n, k):
    """Whether the backend runs these two products as one launch (it does so here, once more)."""
    at = lambda t: None if t is None else t.device_ptr(False)  # noqa: E731
    op = {"gate": ("silu", "mul"), "add first": ("silu", "add"), "others": ("div", "exp"), "plain": (None, None)}[form]
    op = [G.KN_OP.get(name, 0) for name in op]
    first = MatmulOut(at(B), at(C), op[0], int(form == "others"), at(X) if form == "others" else None, at(E))
    second = MatmulOut(at(B2), at(C2), op[1], int(form == "gate"), at({"gate": E, "add first": C}.get(form)), at(E2))
    taken = ctypes.c_int(-1)
    rc = N.backend().mi355_f16_matmul_two(at(A), int(A.column_major), int(B.column_major), b, m, n, k, ctypes.byref(first),
                                          ctypes.byref(second), ctypes.byref(taken))
    assert rc == 0, N.last_error()
    return taken.value


def _check(rt, b, m, n, k, order, form, a_order=ROW, ins=None, finite=True, taken=None):
    g = G.KNGraph()
    try:
        A = g.new_input((b, m, k), layout=a_order)
        B, B2 = (g.new_input((b, k, n), layout=order) for _ in range(2))
        X = g.new_input((b, m, n))
        C = g.matmul(A, B)
        E = g._unary("silu", C) if form in ("gate", "add first") else g.div(X, C) if form == "others" else None
        C2 = g.matmul(A, B2)
        E2 = {"gate": lambda: g._binary("mul", E, C2), "add first": lambda: g._binary("add", C2, C),
              "others": lambda: g._unary("exp", C2), "plain": lambda: None}[form]()
        if ins is None:
            ins = [normal_f16([b, m, k], 0.2, 1), normal_f16([b, k, n], 0.2, 2), normal_f16([b, k, n], 0.2, 3),
                   np.abs(normal_f16([b, m, n], 1.0, 4)) + np.float16(0.5)]
        for t, a in zip((A, B, B2, X), ins):
            t.write_data(a)
        made = [t for t in (C, E, C2, E2) if t is not None]
        for _ in range(2):
            for t in made:
                t.write_data(np.full(t.dims, -7, np.float16))
            g.execute_all()
        got = [t.read_data() for t in made]
        if taken is not None:
            assert _taken(A, B, B2, X, C, E, C2, E2, form, b, m, n, k) == taken
        if finite:
            what = f"{b} x {m} x {k} x {n} {order} {form}"
            assert_f16_close(got[0], orc.f16_matmul(ins[0], ins[1]), what=what)
            assert_f16_close(got[made.index(C2)], orc.f16_matmul(ins[0], ins[2]), what=what)
        for i in range(g.num_operators):  # the consumers again, of the products as they are
            if g.op_type(i) not in (1001, 1003):
                g.execute(i)
        for t, w in zip(made, got):
            np.testing.assert_array_equal(t.read_data().view(np.uint16), w.view(np.uint16))
        return got
    finally:
        g.close()


# batch, m, n, k, weights, input: workgroups of both products, with 64 columns of each and 128, one row of a tile and
# one past it; the three kernels whole and in ranges of k; odd sizes, a column-major input; shapes that go one by one
SHAPES = [(1, 1, 8, 64, ROW, ROW), (1, 65, 72, 192, ROW, ROW), (1, 64, 513, 128, COL, ROW), (1, 385, 2440, 64, ROW, ROW),
          (1, 300, 3332, 128, COL, ROW), (1, 300, 1032, 1024, COL, ROW), (1, 3, 7, 515, COL, ROW), (1, 17, 130, 65, ROW, ROW),
          (1, 33, 513, 1030, ROW, ROW), (1, 5, 72, 1024, ROW, ROW), (1, 130, 72, 1024, COL, ROW), (2, 33, 256, 128, ROW, ROW),
          (1, 40, 72, 520, COL, COL), (1, 257, 1032, 8, COL, COL), (1, 1, 1, 1, COL, ROW)]
# what these are given (test_gemm_choice.py): columns of both in a workgroup, or a kind of tile and its k ranges, or None:
# where the second's consumer reads nothing of the first's, and where it does
STAGED, DIRECT, WAVES = 0, 1, 2
TAKEN = [((STAGED, 1), 64), ((STAGED, 1), 64), ((STAGED, 1), 64), (128, 128), (128, 128), ((DIRECT, 1), 64), ((STAGED, 1), (STAGED, 2)),
         ((STAGED, 1), None), ((STAGED, 1), (STAGED, 4)), ((WAVES, 1), (STAGED, 4)), ((WAVES, 1), (STAGED, 4)), (None, None),
         ((STAGED, 1), (STAGED, 4)), ((STAGED, 1), None), (None, None)]


@pytest.mark.parametrize("form", ["gate", "add first", "others", "plain"])
@pytest.mark.parametrize("b,m,n,k,order,a_order", SHAPES)
def test_two_matmuls_of_one_input(rt, b, m, n, k, order, a_order, form):
    route = TAKEN[SHAPES.index((b, m, n, k, order, a_order))][form in ("gate", "add first")]
    _check(rt, b, m, n, k, order, form, a_order, taken=int(route is not None))


@pytest.mark.parametrize("m,n,k,order", [(5, 72, 192, ROW), (3, 130, 1030, COL), (385, 2440, 64, ROW)])
def test_infinities_and_nan(rt, m, n, k, order):
    """Where the numbers are past the range of fp16 the consumers see them as the products hold them."""
    rng = np.random.default_rng(7)
    ins = [normal_f16([1, m, k], 0.2, 1), normal_f16([1, k, n], 0.2, 2), normal_f16([1, k, n], 0.2, 3), normal_f16([1, m, n], 1.0, 4)]
    ins[0][0, m - 1, k - 1], ins[1][0, k - 1, 0], ins[2][0, 1, n - 1] = np.inf, -np.inf, np.nan
    ins[1][0, rng.integers(k), 3] = np.float16(6e4)
    got = _check(rt, 1, m, n, k, order, "gate", ins=ins, finite=False)
    for c, w in ((got[0], ins[1]), (got[2], ins[2])):
        with np.errstate(invalid="ignore", over="ignore"):
            want = (ins[0][0].astype(np.float64)[:, :, None] * w[0].astype(np.float64)).sum(1)
        np.testing.assert_array_equal(np.isnan(c[0]), np.isnan(want))
        inf = np.isinf(want)
        np.testing.assert_array_equal(c[0][inf], want[inf])


def test_missing_products_and_place(rt, abi):
    out, taken = MatmulOut(), ctypes.c_int()
    for args in ((None, ctypes.byref(out), ctypes.byref(taken)), (ctypes.byref(out), None, ctypes.byref(taken)),
                 (ctypes.byref(out), ctypes.byref(out), None)):
        assert abi.mi355_f16_matmul_two(None, 0, 0, 1, 16, 64, 64, *args) == -3  # MI355_ERR_INVALID
