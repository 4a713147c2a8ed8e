"""silu of every fp16 value, the same bits wherever it is computed: in the prologue of each fused GEMM
kernel, in the interpreter's statement and in the un-fused operator."""
import numpy as np
import pytest

from attention_superoptimizer_amd import workloads as W

pytestmark = pytest.mark.gpu
ROWS, K = 16, 4096


def _every_value():
    x = np.arange(ROWS * K, dtype=np.uint32).astype(np.uint16).view(np.float16).reshape(ROWS, K).copy()
    x[~np.isfinite(x)] = 0  # (an infinity times the zeros beside the diagonal is no number)
    return x


def _run(rt, spec, ins):
    g, vals = rt.build_from_spec(spec)
    try:
        for i, a in ins.items():
            vals[i][0].write_data(a)
        g.execute_all()
        return vals[-1][0].read_data()
    finally:
        g.close()


# option and value that leads a plan of these tiles to the kernel
KERNELS = {"lanes": (7, 2), "stream or lanes": (7, 0), "stream": (7, 1), "tiles": (9, 1)}


@pytest.mark.parametrize("kt", [64, 256])
@pytest.mark.parametrize("gate", [False, True], ids=["silu", "silu_mul"])
@pytest.mark.parametrize("kernel", KERNELS)
def test_fused_silu_is_the_operators(rt, abi, kernel, gate, kt):
    x, eye = _every_value(), np.eye(K, dtype=np.float16)
    if gate:
        ops = [("tb_silu_op", [(0, 0)]), ("tb_mul_op", [(3, 0), (1, 0)]), ("tb_matmul_op", [(4, 0), (2, 0)])]
        plan = W._plan((K // 64, 1, 1), K // kt, [(-1, -1, -1), (-1, -1, -1), (1, -1, -1)], (1, 1, 0), (1, -1, -1), ops)
        spec = [W._inp([ROWS, K]), W._inp([ROWS, K]), W._inp([K, K], "DmemColumnMajor"),
                {"op": "customized", "in": [[0, 0], [1, 0], [2, 0]], "plan": plan}]
        ins = {0: x, 1: np.ones_like(x), 2: eye}
    else:
        ops = [("tb_silu_op", [(0, 0)]), ("tb_matmul_op", [(2, 0), (1, 0)])]
        plan = W._plan((K // 64, 1, 1), K // kt, [(-1, -1, -1), (1, -1, -1)], (1, 0), (1, -1, -1), ops)
        spec = [W._inp([ROWS, K]), W._inp([K, K], "DmemColumnMajor"), {"op": "customized", "in": [[0, 0], [1, 0]], "plan": plan}]
        ins = {0: x, 1: eye}
    alone = _run(rt, [W._inp([ROWS, K]), {"op": "silu", "in": [[0, 0]]}], {0: x})
    option, value = KERNELS[kernel]
    assert abi.mi355_set_option(option, value) == 0
    try:
        fused = _run(rt, spec, ins)
    finally:
        assert abi.mi355_set_option(option, 0) == 0
    assert abi.mi355_set_option(1, 1) == 0
    try:
        interpreted = _run(rt, spec, ins)
    finally:
        assert abi.mi355_set_option(1, 0) == 0
    # (a product's sum starts from +0: the sign of a zero is not kept)
    np.testing.assert_array_equal(interpreted, alone)
    np.testing.assert_array_equal(fused, alone)
