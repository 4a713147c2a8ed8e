"""A gated MLP's two operators (KNGraph.execute_all): the first's kernel leaves silu(G) * U for the second, and every
tensor is bit for bit what the two operators give one by one -- on each kernel that does so, and on those that do not.
Which way was taken shows in the second's launch: a plain product has other LDS sizes than one with silu(a) * u."""
import ctypes

import numpy as np
import pytest

from attention_superoptimizer_amd import _native as N
from attention_superoptimizer_amd import workloads as W
from helpers import normal_f16

pytestmark = pytest.mark.gpu
ROW, COL = "DmemRowMajor", "DmemColumnMajor"


def _last_launch():
    info = N.Mi355LaunchInfo()
    assert N.backend().mi355_last_launch(ctypes.byref(info)) == 0
    return [getattr(info, name) for name, _ in info._fields_]


def _check(rt, spec, order, std, shared, passes=2):
    spec = [dict(op, layout=order) if op["op"] == "input" and op["layout"] == COL else op for op in spec]
    g, vals = rt.build_from_spec(spec)
    try:
        made = []
        for i, op in enumerate(spec):
            if op["op"] == "input":
                vals[i][0].write_data(normal_f16(op["dims"], std[i], 41 + i))
            else:
                g.execute(i)
                made += vals[i]
        alone = _last_launch()
        want = [t.read_data().view(np.uint16) for t in made]
        nan = [np.isnan(t.view(np.float16)) for t in want]
        for _ in range(passes):
            for t in made:
                t.write_data(np.full(t.dims, -7, np.float16))
            g.execute_all()
            assert (_last_launch() != alone) == shared
            for t, w, n in zip(made, want, nan):
                got = t.read_data().view(np.uint16)
                np.testing.assert_array_equal(np.isnan(got.view(np.float16)), n)
                np.testing.assert_array_equal(np.where(n, 0, got), np.where(n, 0, w))
        return made[-1].read_data()
    finally:
        g.close()


def _spec(m, d, h, kt1, kt2):
    return W.config5_gated_mlp(m=m, d=d, h=h, grid1=h // 64, F1=d // kt1, grid2=d // 64, F2=h // kt2)[0]


# rows, d, h, k of the iterations: strips of both weights (8 columns of each), the one-launch kernel, both weights in a
# workgroup (row-major, more than half the chip), ranges and their fold (few blocks, 16 rows), whole blocks of one
# weight; more iterations than the fold's LDS holds (separate operators)
SHAPES = [(8, 512, 2048, 256, 256), (1, 256, 1792, 64, 64), (16, 384, 4096, 128, 128), (9, 192, 1600, 64, 64), (8, 256, 320, 64, 64),
          (16, 512, 448, 128, 64), (8, 704, 129 * 64, 64, 64), (16, 256, 256 * 64, 64, 256), (16, 4096, 512, 64, 64), (8, 8192, 2048, 256, 256),
          (8, 512, 8256, 64, 64), (8, 64, 161 * 64, 64, 64), (7, 128, 640, 128, 128), (33, 256, 320, 64, 64)]
SEPARATE = [((8, 512, 8256, 64, 64), ROW), ((8, 64, 161 * 64, 64, 64), COL), ((8, 64, 161 * 64, 64, 64), ROW)]


@pytest.mark.parametrize("order", [COL, ROW])
@pytest.mark.parametrize("m,d,h,kt1,kt2", SHAPES)
def test_same_tensors(rt, m, d, h, kt1, kt2, order):
    shared = ((m, d, h, kt1, kt2), order) not in SEPARATE
    _check(rt, _spec(m, d, h, kt1, kt2), order, {0: 0.25, 1: 0.05, 2: 0.05, 3: 0.05}, shared)


@pytest.mark.parametrize("order", [COL, ROW])
@pytest.mark.parametrize("m,d,h,kt1,kt2", [(8, 512, 2048, 256, 256), (16, 256, 320, 64, 64)])
def test_infinities_and_nan(rt, m, d, h, kt1, kt2, order):
    """Products past fp16's range: silu(-inf) = -0 or NaN, infinity times zero."""
    out = _check(rt, _spec(m, d, h, kt1, kt2), order, {0: 60.0, 1: 60.0, 2: 60.0, 3: 0.05}, True, passes=1)
    assert np.isnan(out).any()


@pytest.mark.parametrize("swap", [False, True])
def test_the_second_operator_names_its_inputs(rt, swap):
    """silu of the first result times the second, or the other way round: only the first way is shared."""
    spec = _spec(8, 256, 320, 64, 64)
    if swap:
        spec[-1] = dict(spec[-1], **{"in": [spec[-1]["in"][1], spec[-1]["in"][0]] + spec[-1]["in"][2:]})
    _check(rt, spec, COL, {0: 0.25, 1: 0.05, 2: 0.05, 3: 0.05}, not swap)
