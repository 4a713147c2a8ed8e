"""A two-output attention operator and the operator behind it that folds its pieces and divides, in one launch
(KNGraph.execute_all): every tensor bit for bit what the two operators give one by one, on every kernel that
folds, where a workgroup has whole rows and where the last of several does, launch after launch."""
import ctypes

import numpy as np
import pytest

from attention_superoptimizer_amd import _native as N
from attention_superoptimizer_amd import workloads as W
from helpers import normal_f16
from test_gpu_f16 import KERNEL_ATTENTION, KERNEL_COMBINE

pytestmark = pytest.mark.gpu
ROW, COL = "DmemRowMajor", "DmemColumnMajor"


def _last_kernel():
    info = N.Mi355LaunchInfo()
    assert N.backend().mi355_last_launch(ctypes.byref(info)) == 0
    return info.kernel_id


def _check(rt, spec, folds, std=0.125, passes=3):
    g, vals = rt.build_from_spec(spec)
    try:
        made = []
        for i, op in enumerate(spec):
            if op["op"] == "input":
                vals[i][0].write_data(normal_f16(op["dims"], std, 31 + i))
            else:
                g.execute(i)
                made += vals[i]
        assert _last_kernel() == KERNEL_COMBINE
        want = [t.read_data().view(np.uint16) for t in made]
        nan = [np.isnan(t.view(np.float16)) for t in want]
        for _ in range(passes):
            for t in made:
                t.write_data(np.full(t.dims, -7, np.float16))
            g.execute_all()
            assert _last_kernel() == (KERNEL_ATTENTION if folds else KERNEL_COMBINE)
            for t, w, n in zip(made, want, nan):
                got = t.read_data().view(np.uint16)
                np.testing.assert_array_equal(np.isnan(got.view(np.float16)), n)
                np.testing.assert_array_equal(np.where(n, 0, got), np.where(n, 0, w))
        return made[-1].read_data()
    finally:
        g.close()


def _decode(groups, rows, keys, blocks, loop, order):
    spec, _ = W.gqa_inc_decode(groups=groups, rows=rows, seq=keys * blocks * loop, kv_blocks=blocks, F=loop)
    return [dict(op, layout=order) if i in (1, 2) else op for i, op in enumerate(spec)]


def _prefill(heads, row_tile, blocks, hd, keys, loop, order, ops=W.COMBINE_OPS, rows2=None):
    tokens, seq = row_tile * blocks, keys * loop
    rows2 = rows2 or (16 if tokens % 16 == 0 else tokens)
    return [W._inp([heads, tokens, hd]), W._inp([heads, hd, seq], order), W._inp([heads, seq, hd], order),
            {"op": "customized", "in": [[0, 0], [1, 0], [2, 0]],
             "plan": W._plan((heads, 1, blocks), loop, [(0, -1, 1), (0, 2, -1), (0, 1, -1)], (-1, 2, 1), (0, 2, 1), W.ATT_OPS, dimx=hd)},
            {"op": "customized", "in": [[3, 0], [3, 1]],
             "plan": W._plan((heads, tokens // rows2, 1), 1, [(0, 1, -1), (0, 1, -1)], (-1, -1), (0, 1, -1), ops, dimx=hd)}]


# groups, rows, key tile, blocks, for-loop, whether one launch folds them: one iteration a wavefront and more, one row
# and parts of a 16-row group, row blocks of several workgroups, two and sixteen pieces; seventeen pieces, blocks that
# do not all run at once and one wavefront for 256 columns are two launches
DECODE = [(2, 8, 64, 16, 4, True), (3, 16, 64, 2, 9, True), (1, 1, 64, 5, 1, True), (2, 64, 64, 3, 8, True), (4, 16, 128, 6, 6, True),
          (3, 16, 32, 4, 4, True), (5, 12, 48, 12, 5, True), (2, 33, 80, 4, 7, True), (1, 1, 48, 4, 15, True), (9, 20, 16, 8, 3, True), (2, 16, 64, 9, 1, False),
          (2, 16, 64, 17, 4, False), (40, 8, 64, 16, 16, False)]


@pytest.mark.parametrize("order", [COL, ROW])
@pytest.mark.parametrize("groups,rows,keys,blocks,loop,folds", DECODE)
def test_pieces_of_several_workgroups(rt, groups, rows, keys, blocks, loop, folds, order):
    _check(rt, _decode(groups, rows, keys, blocks, loop, order), folds)


@pytest.mark.parametrize("groups,rows,keys,blocks,loop,folds", [
    (7, 1, 64, 4, 5, True), (8, 1, 64, 4, 5, False), (8, 1, 64, 5, 5, True), (16, 1, 48, 2, 3, False), (2, 1, 32, 16, 3, False),
    (1, 1, 32, 16, 3, True), (8, 16, 64, 16, 4, True), (9, 16, 64, 16, 4, False), (9, 2, 80, 16, 2, False), (9, 2, 80, 15, 2, True),
    (24, 8, 64, 8, 4, True), (25, 8, 64, 8, 4, False), (25, 8, 64, 9, 4, True), (7, 1, 32, 4, 7, True), (7, 1, 32, 4, 8, False),
    (5, 1, 32, 4, 13, True), (6, 1, 32, 4, 13, False), (18, 1, 32, 5, 7, True), (18, 1, 32, 5, 16, False), (9, 1, 32, 5, 16, True),
    (6, 1, 16, 8, 11, False), (5, 1, 16, 8, 11, True), (16, 1, 32, 3, 8, False), (15, 1, 32, 3, 8, True), (21, 1, 32, 7, 12, True),
    (7, 2, 32, 4, 13, True)])
def test_where_the_other_launch_is_short(rt, groups, rows, keys, blocks, loop, folds):
    """Few pieces of one row, and sixteen of more: two launches from so many workgroups on, fewer in long loops."""
    _check(rt, _decode(groups, rows, keys, blocks, loop, ROW), folds)


# heads, row tile, row blocks, head size, key tile, for-loop: the streaming kernel (128- and 64-row slabs, 256-row
# ones, wide key tiles), the one for whole tiles, the one with a tile pair a wavefront, the one for any size
PREFILL = [(16, 128, 32, 64, 64, 4), (32, 128, 16, 128, 64, 2), (32, 64, 16, 64, 64, 3), (4, 256, 130, 64, 64, 2), (4, 128, 8, 128, 256, 2),
           (3, 32, 3, 128, 64, 5), (2, 128, 2, 64, 256, 1), (2, 80, 5, 64, 64, 31), (2, 32, 7, 64, 64, 3), (3, 32, 4, 64, 32, 22),
           (12, 80, 13, 64, 80, 13), (2, 48, 5, 128, 48, 3), (2, 24, 3, 64, 16, 5)]


@pytest.mark.parametrize("order", [COL, ROW])
@pytest.mark.parametrize("shape", PREFILL)
def test_whole_rows(rt, shape, order):
    _check(rt, _prefill(*shape, order), True)


@pytest.mark.parametrize("ops,folds", [
    ([("tb_reduction_2_op", [(1, 0)]), ("tb_div_op", [(0, 0), (2, 0)])], True),
    ([("tb_div_op", [(0, 0), (1, 0)])], True),
    ([("tb_reduction_2_op", [(1, 0)]), ("tb_div_op", [(0, 0), (2, 0)]), ("tb_reduction_2_to_dimx_op", [(3, 0)])], True)])
def test_places_of_the_division(rt, ops, folds):
    """With one piece a row every place of the division comes to the same."""
    _check(rt, _prefill(2, 64, 3, 64, 64, 5, COL, ops), folds)


@pytest.mark.parametrize("order", [COL, ROW])
@pytest.mark.parametrize("shape", [(2, 64, 3, 64, 64, 5), (3, 48, 3, 64, 48, 7), (16, 128, 32, 64, 64, 4), (2, 64, 3, 128, 64, 3)])
@pytest.mark.parametrize("ops,sign", [
    (W.COMBINE_OPS, True),
    ([("tb_reduction_2_op", [(1, 0)]), ("tb_div_op", [(0, 0), (2, 0)])], False),
    ([("tb_div_op", [(0, 0), (1, 0)])], False),
    ([("tb_reduction_2_op", [(1, 0)]), ("tb_div_op", [(0, 0), (2, 0)]), ("tb_reduction_2_to_dimx_op", [(3, 0)])], False)])
def test_signs_of_zero(rt, ops, sign, shape, order):
    """Negative numerators over infinite row sums: the quotient is -0, and stays it where nothing is added to it
    behind the division; a sum or a saver behind it begins with +0.  On every kernel that divides as it stores."""
    out = _check(rt, _prefill(*shape, order, ops), True, std=0.7, passes=1).view(np.uint16)
    assert (out == 0).any() and (out == 0x8000).any() == sign


@pytest.mark.parametrize("spec", [_decode(2, 16, 64, 4, 4, COL), _prefill(4, 128, 2, 64, 64, 4, COL), _prefill(3, 48, 3, 64, 48, 3, ROW)])
def test_infinities_and_nan(rt, spec):
    """Scores past the exponential's range: infinite row sums, infinity over infinity, zero over zero."""
    out = _check(rt, spec, True, std=4.0, passes=1)
    assert np.isnan(out).any()
