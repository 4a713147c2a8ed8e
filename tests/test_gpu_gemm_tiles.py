"""The skinny-GEMM kernel for tiles of any size against the fp16 oracle: activation tiles around the
edges of a 16-row group and of a row slab, weight tiles of 16 / 48 / 128 columns, iterations of one
step of 32 k and of more steps than are in flight together, fewer and more iterations than lanes
and than a round holds, every member of the family, every LoRA rank, both storage orders."""
import pytest

from helpers import assert_f16_close, normal_f16
from oracle import evaluate as orc
from test_gpu_f16 import KERNEL_GEMM, _graph_f16, _last_kernels

pytestmark = pytest.mark.gpu
ROW, COL = "DmemRowMajor", "DmemColumnMajor"


@pytest.fixture
def any_size_kernel(abi):
    assert abi.mi355_set_option(9, 1) == 0
    yield
    assert abi.mi355_set_option(9, 0) == 0


def _run(rt, spec, order, what, std=0.1):
    spec = [dict(op, layout=order) if op["op"] == "input" and i > 0 else op for i, op in enumerate(spec)]
    # (weights of one sign: no cancellation between iterations)
    ins = {i: normal_f16(op["dims"], std, 5 + i) for i, op in enumerate(spec) if op["op"] == "input"}
    ins = {i: abs(a) if i in (0, 1) else a for i, a in ins.items()}
    got = _graph_f16(rt, spec, ins)
    want = orc.eval_graph(spec, "f16", ins, threads=8)
    for i, op in enumerate(spec):
        if op["op"] == "customized":
            for j, w in enumerate(want[i]):
                assert_f16_close(got[i][j], w, what=f"{what} op {i} out {j}")
    assert _last_kernels == [KERNEL_GEMM] * len(_last_kernels), what


@pytest.mark.parametrize("order", [COL, ROW])
@pytest.mark.parametrize("m,cols,blocks,kt,loop", [
    (1, 16, 3, 32, 5), (15, 48, 5, 96, 8), (17, 128, 4, 288, 9), (64, 64, 3, 320, 3), (65, 32, 2, 64, 40),
    (200, 32, 70, 64, 2), (33, 128, 150, 32, 17), (64, 64, 2, 32, 130)])
def test_plain(rt, any_size_kernel, m, cols, blocks, kt, loop, order):
    from attention_superoptimizer_amd import workloads as W
    spec, _ = W.tiled_matmul(m, cols * blocks, kt * loop, (blocks, 1, 1), loop, (-1, -1, -1), (1, -1, -1), (1, -1, -1))
    _run(rt, spec, order, f"{m} x {cols} x {blocks}, {kt} x {loop} {order}")


@pytest.mark.parametrize("order", [COL, ROW])
@pytest.mark.parametrize("m", [1, 9, 16, 30])
def test_gated_mlp_and_prologues(rt, any_size_kernel, m, order):
    from attention_superoptimizer_amd import workloads as W
    spec, _ = W.config5_gated_mlp(m=m, d=192, h=320, grid1=5, F1=2, grid2=3, F2=5)
    _run(rt, spec, order, f"gated mlp {m} {order}", std=0.05)
    for op in ("tb_exp_op", "tb_silu_op"):
        spec = [W._inp([m, 160]), W._inp([160, 96], COL),
                {"op": "customized", "in": [[0, 0], [1, 0]],
                 "plan": W._plan((2, 1, 1), 5, [(-1, -1, -1), (1, -1, -1)], (1, 0), (1, -1, -1),
                                 [(op, [(0, 0)]), ("tb_matmul_op", [(2, 0), (1, 0)])])}]
        _run(rt, spec, order, f"{op} {m} {order}")


@pytest.mark.parametrize("order", [COL, ROW])
@pytest.mark.parametrize("m,rank,kt", [(1, 8, 64), (16, 16, 256), (13, 32, 160), (31, 8, 32), (32, 32, 128)])
def test_lora(rt, any_size_kernel, m, rank, kt, order):
    from attention_superoptimizer_amd import workloads as W
    spec, _ = W.config4_lora(m=m, d=kt * 3, r=rank, grid=3, F=3)
    spec[1], spec[3] = W._inp([kt * 3, 192], COL), W._inp([rank, 192], COL)
    _run(rt, spec, order, f"lora {m} rank {rank} {kt} {order}")
