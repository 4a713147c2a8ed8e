"""The un-fused attention graph in one launch (mi355_f16_attention_rows): every one of its tensors."""
import ctypes

import numpy as np
import pytest

from attention_superoptimizer_amd import graph as G
from attention_superoptimizer_amd import workloads as W
from helpers import normal_f16

pytestmark = pytest.mark.gpu

ULP = 2.0 ** -11        # one rounding to fp16, relative
SMALL = 2.0 ** -24      # the spacing of subnormal fp16 numbers


def _run(abi, b, m, n, d, order, ins, taken):
    """The five tensors as a graph leaves them; the entry point by itself, first, has to say `taken` and, where
    it does, to leave the same."""
    spec = W.attention_reference([b, m, d], [b, d, n], [b, n, d])
    spec[1], spec[2] = dict(spec[1], layout=order), dict(spec[2], layout=order)
    g, t = G.build_from_spec(spec)
    try:
        for i, a in enumerate(ins):
            t[i][0].write_data(a)

        def poison():  # (nothing that an earlier run left is taken for a result)
            for i in range(3, 8):
                t[i][0].write_data(np.full(spec_dims(t[i][0]), 7, np.float16))

        poison()
        answer = ctypes.c_int(7)
        assert abi.mi355_f16_attention_rows(*[t[i][0].device_ptr(False) for i in range(8)], b, m, n, d, d,
                                            1 if order == "DmemColumnMajor" else 0, ctypes.byref(answer)) == 0
        assert answer.value == taken
        alone = [t[i][0].read_data() for i in range(3, 8)]
        poison()
        g.execute_all()
        got = [t[i][0].read_data() for i in range(3, 8)]
        for x, y in zip(alone, got):
            np.testing.assert_array_equal(x, y if taken else 7)
        return got
    finally:
        g.close()


def spec_dims(t):
    return tuple(t.dims)


def _check(ins, got):
    """Each tensor against its operator on the tensors before it: fp32 sums of products (error below
    2^-22 of the terms' magnitudes for these lengths), then one rounding."""
    q, k, v = (x.astype(np.float64) for x in ins)
    s, e, r, p, o = (x.astype(np.float64) for x in got)
    want, terms = np.matmul(q, k), np.matmul(np.abs(q), np.abs(k))
    assert np.all(np.abs(s - want) <= ULP * np.abs(want) + 2.0 ** -20 * terms + SMALL)
    want = np.exp(s)
    assert np.all(np.abs(e - want) <= (ULP + 1e-5) * want + SMALL)  # (exp in fp32: arguments up to 16)
    want = e.sum(-1, keepdims=True)
    assert np.all(np.abs(r - want) <= (ULP + 1e-5) * want)
    np.testing.assert_array_equal(got[3], (got[1].astype(np.float32) / got[2].astype(np.float32)).astype(np.float16))
    want, terms = np.matmul(p, v), np.matmul(p, np.abs(v))
    assert np.all(np.abs(o - want) <= ULP * np.abs(want) + 2.0 ** -20 * terms + SMALL)


@pytest.mark.parametrize("order", ["DmemRowMajor", "DmemColumnMajor"])
@pytest.mark.parametrize("b,m,n,d,taken", [
    (1, 1, 32, 64, 1),      # the smallest
    (3, 17, 33, 128, 1),    # one row past a block of rows, one key past a block of keys
    (2, 15, 255, 64, 1),
    (1, 16, 257, 128, 1),   # one key into the wavefronts' second blocks
    (9, 33, 500, 64, 1),
    (2, 40, 767, 64, 1),    # three blocks each
    (2, 20, 700, 128, 1),
    (2, 40, 801, 128, 0),   # too few workgroups for a row of four blocks each
    (22, 40, 801, 128, 1),  # enough
    (3, 40, 1024, 64, 1),
    (1, 20, 1500, 64, 1),
    (1, 300, 2047, 64, 1),  # sixteen wavefronts with four blocks each
    (129, 7, 1100, 128, 1),
    (130, 3, 2048, 128, 1),
    (1, 33, 2049, 64, 0),   # too long for one launch
])
def test_every_tensor(rt, abi, order, b, m, n, d, taken):
    ins = [normal_f16([b, m, d], 0.3, 1), normal_f16([b, d, n], 0.3, 2), normal_f16([b, n, d], 0.5, 3)]
    _check(ins, _run(abi, b, m, n, d, order, ins, taken))


@pytest.mark.parametrize("order", ["DmemRowMajor", "DmemColumnMajor"])
@pytest.mark.parametrize("b,m,n,d,taken", [
    (2, 20, 77, 64, 1),      # (one block of keys a wavefront,
    (2, 33, 1030, 64, 1),    # three,
    (2, 20, 700, 128, 1),    # three, the last one masked,
    (43, 33, 1030, 128, 1),  # six)
    (2, 33, 1030, 128, 0)])  # three launches
def test_numbers_out_of_range_stay_where_they_belong(rt, abi, order, b, m, n, d, taken):
    """Rows and keys with infinities and NaN, at the edges above all: a tensor's non-finite elements are
    those its operator gives on the tensors before it."""
    ins = [normal_f16([b, m, d], 0.3, 1), normal_f16([b, d, n], 0.3, 2), normal_f16([b, n, d], 0.5, 3)]
    ins[0][0, m - 1, d - 1], ins[0][0, 3, 5] = np.nan, np.inf
    ins[1][0, :, n - 1], ins[2][1, n - 1, 2], ins[2][0, 0, d - 1] = 60000, np.nan, np.inf
    ins[0][1, 4, :], ins[1][1, :, 9] = 8, 8  # (a score whose exponential overflows)
    got = _run(abi, b, m, n, d, order, ins, taken)
    with np.errstate(all="ignore"):
        f = [x.astype(np.float32) for x in ins + got]
        wants = [np.matmul(f[0], f[1]), np.exp(f[3]), f[4].sum(-1, keepdims=True), f[4] / f[5], np.matmul(f[6], f[2])]
        for name, x, want in zip("SERPO", got, (w.astype(np.float16) for w in wants)):
            assert np.array_equal(np.isnan(x), np.isnan(want)), name
            assert np.array_equal(np.isinf(x), np.isinf(want)) and np.array_equal(np.signbit(x[np.isinf(x)]),
                                                                                  np.signbit(want[np.isinf(want)])), name


def test_no_place_for_the_answer(abi):
    assert abi.mi355_f16_attention_rows(*[None] * 8, 1, 16, 64, 64, 64, 0, None) != 0
