"""The fold-and-divide operators of split attention plans as fingerprints: one launch without tiles in LDS, the
interpreter's values bit for bit."""
import numpy as np
import pytest

from helpers import uniform_fp
from test_gpu_fingerprint import _graph_fp
from test_gpu_launch_records import _kernel as launched

pytestmark = pytest.mark.gpu
KERNEL_FP_INTERP, KERNEL_FP_COMBINE = 1, 8


def _spec(kind, rows, pieces, x, dens, loop, grid):
    from attention_superoptimizer_amd import workloads as W
    ops = {"sum, divide": [("tb_reduction_2_to_dimx_op", [(0, 0)]), ("tb_reduction_2_op", [(1, 0)]), ("tb_div_op", [(2, 0), (3, 0)])],
           "sum, divide by one": [("tb_reduction_2_to_dimx_op", [(0, 0)]), ("tb_div_op", [(2, 0), (1, 0)])],
           "divide, sum": [("tb_reduction_2_op", [(1, 0)]), ("tb_div_op", [(0, 0), (2, 0)]), ("tb_reduction_2_to_dimx_op", [(3, 0)])],
           "divide, accumulate": [("tb_reduction_2_op", [(1, 0)]), ("tb_div_op", [(0, 0), (2, 0)])]}[kind]
    plan = W._plan(grid, loop, [(0, 1, -1), (0, 1, -1)], (2 if loop > 1 else -1, -1), (0, 1, -1), ops)
    plan["reduction_dimx"] = x
    return [W._inp([grid[0], grid[1] * rows, pieces * x]), W._inp([grid[0], grid[1] * rows, dens]), {"op": "customized", "in": [[0, 0], [1, 0]], "plan": plan}]


@pytest.mark.parametrize("kind,rows,pieces,x,dens,loop", [
    ("sum, divide", 8, 4, 64, 4, 1), ("sum, divide", 1, 1, 8, 1, 1), ("sum, divide", 33, 7, 24, 5, 1), ("sum, divide", 5, 17, 4, 9, 1),
    ("sum, divide by one", 16, 3, 32, 1, 1), ("divide, sum", 7, 6, 64, 3, 1), ("divide, sum", 3, 5, 12, 2, 1),
    ("divide, accumulate", 9, 1, 64, 4, 1), ("divide, accumulate", 9, 4, 16, 4, 4),
    ("divide, accumulate, many blocks", 5, 4, 16, 4, 4), ("divide, accumulate, many blocks", 1, 3, 12, 1, 3)])
def test_fold_and_divide_equals_the_interpreter(rt, abi, kind, rows, pieces, x, dens, loop):
    grid = (8, 24, 1) if "many blocks" in kind else (2, 3, 1)
    spec = _spec(kind.replace(", many blocks", ""), rows, pieces, x, dens, loop, grid)
    ins = {i: uniform_fp(spec[i]["dims"], 40 + i) for i in range(2)}
    ins[0].flat[::5] = 65535  # (any 16-bit value is an operand)
    ins[1].flat[::3] = 0      # and a sum that is zero in one ring or both a divisor
    got = _graph_fp(rt, spec, ins)[2][0]
    # (fewer than 192 blocks share the for-loop out, and the interpreter does that)
    split = loop > 1 and grid[0] * grid[1] < 192
    assert launched() == ((KERNEL_FP_INTERP, 6 * loop) if split else (KERNEL_FP_COMBINE, grid[0] * grid[1]))
    assert abi.mi355_set_option(1, 1) == 0
    try:
        want = _graph_fp(rt, spec, ins)[2][0]
        assert launched()[0] == KERNEL_FP_INTERP
    finally:
        assert abi.mi355_set_option(1, 0) == 0
    np.testing.assert_array_equal(got, want)
