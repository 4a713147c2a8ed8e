"""The streaming skinny-GEMM kernel against the fp16 oracle: rows around the edges of a 16-row group,
for-loops of one range and of many (ranges that do not divide by the wavefronts), every member of the
family, both storage orders.  (Option 7 = 1 keeps small plans off the one-launch kernel.)"""
import pytest

from test_gpu_gemm_tiles import COL, ROW, _run

pytestmark = pytest.mark.gpu


@pytest.fixture
def ranges(abi):
    assert abi.mi355_set_option(7, 1) == 0
    yield
    assert abi.mi355_set_option(7, 0) == 0


@pytest.mark.parametrize("order", [COL, ROW])
@pytest.mark.parametrize("m,blocks,kt,loop", [
    (1, 100, 64, 7), (16, 3, 64, 1), (17, 5, 64, 9), (15, 2, 512, 6), (33, 4, 128, 30), (64, 3, 128, 5), (4, 300, 64, 20),
    (2, 1, 64, 200)])
def test_plain(rt, ranges, m, blocks, kt, loop, order):
    from attention_superoptimizer_amd import workloads as W
    spec, _ = W.tiled_matmul(m, 64 * blocks, kt * loop, (blocks, 1, 1), loop, (-1, -1, -1), (1, -1, -1), (1, -1, -1))
    _run(rt, spec, order, f"{m} x {blocks}, {kt} x {loop} {order}")


@pytest.mark.parametrize("order", [COL, ROW])
@pytest.mark.parametrize("m", [1, 9, 16])
def test_gated_mlp_prologues_and_lora(rt, ranges, m, order):
    from attention_superoptimizer_amd import workloads as W
    spec, _ = W.config5_gated_mlp(m=m, d=192, h=640, grid1=10, F1=3, grid2=3, F2=5)
    _run(rt, spec, order, f"gated mlp {m} {order}", std=0.05)
    for op in ("tb_exp_op", "tb_silu_op"):
        spec = [W._inp([m, 320]), W._inp([320, 128], COL),
                {"op": "customized", "in": [[0, 0], [1, 0]],
                 "plan": W._plan((2, 1, 1), 5, [(-1, -1, -1), (1, -1, -1)], (1, 0), (1, -1, -1),
                                 [(op, [(0, 0)]), ("tb_matmul_op", [(2, 0), (1, 0)])])}]
        _run(rt, spec, order, f"{op} {m} {order}")
    spec, _ = W.config4_lora(m=m, d=128 * 6, r=16, grid=3, F=6)
    spec[1], spec[3] = W._inp([128 * 6, 192], COL), W._inp([16, 192], COL)
    _run(rt, spec, order, f"lora {m} {order}")


@pytest.mark.parametrize("order", [COL, ROW])
@pytest.mark.parametrize("option,value", [(7, 1), (7, 2), (9, 1)], ids=["stream", "lanes", "tiles"])
@pytest.mark.parametrize("family", ["plain", "silu", "exp", "gated", "lora"])
def test_infinities_and_nan(rt, abi, family, option, value, order):
    """Infinities, NaN, prologues that overflow and sums that do, in the first and last rows, columns and
    iterations: the interpreter's pattern, and its numbers where they are finite."""
    import numpy as np
    from attention_superoptimizer_amd import workloads as W
    from helpers import assert_f16_close, normal_f16
    from test_gpu_f16 import _graph_f16
    m = 9
    if family == "gated":
        spec, _ = W.config5_gated_mlp(m=m, d=192, h=640, grid1=10, F1=3, grid2=3, F2=5)
    elif family == "lora":
        spec, _ = W.config4_lora(m=m, d=128 * 6, r=16, grid=3, F=6)
        spec[1], spec[3] = W._inp([128 * 6, 192], COL), W._inp([16, 192], COL)
    else:
        ops = [("tb_matmul_op", [(0, 0), (1, 0)])] if family == "plain" else [
            (f"tb_{family}_op", [(0, 0)]), ("tb_matmul_op", [(2, 0), (1, 0)])]
        spec = [W._inp([m, 320]), W._inp([320, 128], COL),
                {"op": "customized", "in": [[0, 0], [1, 0]],
                 "plan": W._plan((2, 1, 1), 5, [(-1, -1, -1), (1, -1, -1)], (1, 0), (1, -1, -1), ops)}]
    spec = [dict(op, layout=order) if op["op"] == "input" and i > 0 else op for i, op in enumerate(spec)]
    ins = {i: normal_f16(op["dims"], 0.1, 5 + i) for i, op in enumerate(spec) if op["op"] == "input"}
    x, w = ins[0], ins[1]
    x[0, 0], x[2, 5], x[3, 7], x[m - 1, -1] = np.inf, np.nan, 60000, -np.inf
    w[3, 1], w[-1, -1], w[0, 4] = np.inf, np.nan, 50000
    got = {}
    for name, (o, v) in {"fused": (option, value), "interpreter": (1, 1)}.items():
        assert abi.mi355_set_option(o, v) == 0
        try:
            got[name] = [t for i, r in enumerate(_graph_f16(rt, spec, ins)) if spec[i]["op"] == "customized" for t in r]
        finally:
            assert abi.mi355_set_option(o, 0) == 0
    for i, (f, want) in enumerate(zip(got["fused"], got["interpreter"])):
        assert np.array_equal(np.isnan(f), np.isnan(want)) and np.array_equal(np.isposinf(f), np.isposinf(want))
        ok = np.isfinite(want)
        assert not ok.all() and (ok.any() or i > 0)  # (a NaN column of the first operator is in all sums of a second)
        assert_f16_close(f[ok], want[ok], what=family)


@pytest.mark.parametrize("order", [COL, ROW])
@pytest.mark.parametrize("m,blocks,kt,loop", [
    (64, 25, 256, 3), (49, 97, 128, 9), (33, 25, 64, 17), (1, 97, 256, 9), (17, 9, 256, 16), (7, 385, 64, 2)])
def test_one_launch_of_many_pieces(rt, abi, m, blocks, kt, loop, order):
    """The one-launch kernel around its line between 16 and 8 wavefronts a workgroup (pieces x k = 98304),
    with loops that its wavefronts do not divide and rows around the edges of 16."""
    from attention_superoptimizer_amd import workloads as W
    spec, _ = W.tiled_matmul(m, 64 * blocks, kt * loop, (blocks, 1, 1), loop, (-1, -1, -1), (1, -1, -1), (1, -1, -1))
    assert abi.mi355_set_option(7, 2) == 0
    try:
        _run(rt, spec, order, f"pieces {m} x {blocks}, {kt} x {loop} {order}")
    finally:
        assert abi.mi355_set_option(7, 0) == 0


@pytest.mark.parametrize("weights", [1, 2])
@pytest.mark.parametrize("m,blocks,kt,loop", [
    (1, 48, 64, 1), (8, 50, 64, 3), (9, 49, 192, 5), (16, 96, 128, 10), (7, 48, 512, 2), (4, 200, 64, 33), (16, 48, 64, 24)])
def test_strips_of_16_columns(rt, ranges, m, blocks, kt, loop, weights):
    """Column-major plans wide enough for a workgroup per 16 columns: rows around 8 and 16, loops that leave
    wavefronts with no, one or fewer iterations, a first step that is also the last, up to the most results that
    fit (16 rows, 24 iterations)."""
    from attention_superoptimizer_amd import workloads as W
    if weights == 1:
        spec, _ = W.tiled_matmul(m, 64 * blocks, kt * loop, (blocks, 1, 1), loop, (-1, -1, -1), (1, -1, -1), (1, -1, -1))
    else:
        # (the first operator alone: the second adds up to 200 products of both signs in an fp16 accumulator that
        # passes 4, where one rounding is 0.004, and ends near 0.3, whose plain bar is 0.004)
        spec, _ = W.config5_gated_mlp(m=m, d=kt * loop, h=64 * blocks, grid1=blocks, F1=loop, grid2=kt * loop // 64, F2=blocks)
        spec = [op for i, op in enumerate(spec[:5]) if i != 3]
    _run(rt, spec, COL, f"strips {m} x {blocks}, {kt} x {loop}, {weights}", **({} if weights == 1 else {"std": 0.05}))


@pytest.mark.parametrize("family,m,blocks,loop", [
    ("plain", 9, 49, 7), ("plain", 16, 63, 3), ("plain", 15, 51, 33), ("plain", 16, 49, 56), ("plain", 7, 51, 53),
    ("lora", 1, 41, 3), ("lora", 8, 63, 17), ("lora", 7, 49, 56), ("lora", 9, 41, 7), ("lora", 16, 63, 4), ("lora", 15, 51, 33)])
def test_one_strip_a_compute_unit(rt, abi, family, m, blocks, loop):
    """256-k iterations whose strips are at most one to a compute unit, on the ordinary rule: rows around 8 and 16, a
    for-loop that the wavefronts share evenly and not, the fewest and many results; against the oracle, and bit for bit
    what the one-launch kernel gives, infinities and NaN included."""
    import numpy as np
    from attention_superoptimizer_amd import workloads as W
    from helpers import normal_f16
    from test_gpu_f16 import _graph_f16
    from test_gpu_launch_records import _kernel as launched
    k, n = 256 * loop, 64 * blocks
    if family == "lora":
        spec, _ = W.config4_lora(m=m, d=k, r=16, grid=blocks, F=loop)
        spec[1], spec[3] = W._inp([k, n], COL), W._inp([16, n], COL)
    else:
        spec, _ = W.tiled_matmul(m, n, k, (blocks, 1, 1), loop, (-1, -1, -1), (1, -1, -1), (1, -1, -1))
    _run(rt, spec, COL, f"lone strips {family} {m} x {blocks}, {loop}", std=0.03)
    assert launched()[1] == 4 * blocks
    ins = {i: normal_f16(op["dims"], 1.0, 9 + i) for i, op in enumerate(spec) if op["op"] == "input"}
    ins[0][m - 1, k - 1], ins[1][5, n - 1], ins[1][k - 3, 17] = np.inf, np.nan, -np.inf
    want = None
    for option in (0, 2):
        assert abi.mi355_set_option(7, option) == 0
        try:
            got = _graph_f16(rt, spec, ins)[-1][0]
        finally:
            assert abi.mi355_set_option(7, 0) == 0
        nan = np.isnan(got)
        bits = np.where(nan, 0, got.view(np.uint16))
        if want is not None:
            np.testing.assert_array_equal(nan, want[0])
            np.testing.assert_array_equal(bits, want[1])
        want = (nan, bits)


@pytest.mark.parametrize("order", [COL, ROW])
@pytest.mark.parametrize("m,cols,blocks,kt,loop,rank", [
    (1, 16, 9, 64, 3, 0), (33, 48, 3, 128, 5, 0), (64, 128, 7, 256, 9, 0), (17, 80, 2, 64, 17, 0), (9, 32, 65, 256, 2, 0),
    (1, 64, 5, 96, 4, 0), (50, 48, 3, 32, 18, 0), (16, 16, 9, 96, 1, 0), (3, 64, 4, 96, 6, 16), (20, 32, 3, 32, 5, 32),
    (17, 64, 3, 64, 4, 16), (5, 64, 9, 256, 9, 32), (33, 32, 5, 128, 3, 32), (16, 64, 2, 64, 17, 8), (64, 16, 3, 256, 2, 8)])
def test_one_launch_of_any_columns_and_rank(rt, abi, m, cols, blocks, kt, loop, rank, order):
    """The one-launch kernel on blocks of one and more 16-column pieces, of several 16-row pieces, with a lora A
    of half a piece (column-major; left to the tiles row-major) and of two."""
    from attention_superoptimizer_amd import workloads as W
    if rank == 0:
        spec, _ = W.tiled_matmul(m, cols * blocks, kt * loop, (blocks, 1, 1), loop, (-1, -1, -1), (1, -1, -1), (1, -1, -1))
    else:
        spec, _ = W.config4_lora(m=m, d=kt * loop, r=rank, grid=blocks, F=loop)
        spec[1], spec[3] = W._inp([kt * loop, cols * blocks], COL), W._inp([rank, cols * blocks], COL)
    assert abi.mi355_set_option(7, 2) == 0
    try:
        _run(rt, spec, order, f"pieces {m} x {cols} x {blocks}, {kt} x {loop}, rank {rank} {order}")
    finally:
        assert abi.mi355_set_option(7, 0) == 0


@pytest.mark.parametrize("order", [COL, ROW])
@pytest.mark.parametrize("option", [0, 1, 2], ids=["rule", "stream", "lanes"])
@pytest.mark.parametrize("m,loop1,loop2", [(1, 9, 17), (16, 13, 8), (8, 17, 41), (9, 64, 2)])
def test_two_weights_uneven_rounds(rt, abi, m, loop1, loop2, option, order):
    """Loops that do not divide by a workgroup's wavefronts, and ranges of 8 iterations whose last one is short."""
    from attention_superoptimizer_amd import workloads as W
    spec, _ = W.config5_gated_mlp(m=m, d=64 * loop1, h=64 * loop2, grid1=loop2, F1=loop1, grid2=loop1, F2=loop2)
    assert abi.mi355_set_option(7, option) == 0
    try:
        _run(rt, spec, order, f"{m} x {64 * loop1} x {64 * loop2} {order}", std=0.02)
    finally:
        assert abi.mi355_set_option(7, 0) == 0


@pytest.mark.parametrize("order", [COL, ROW])
@pytest.mark.parametrize("family", ["exp", "silu", "silu_mul"])
@pytest.mark.parametrize("m,cols,blocks,kt,loop,extremes", [
    (17, 16, 9, 32, 5, False), (33, 48, 3, 96, 4, False), (64, 64, 2, 96, 3, False), (64, 48, 5, 32, 17, False),
    (33, 64, 2, 64, 6, False), (17, 64, 9, 256, 2, False), (49, 16, 3, 128, 5, False),
    (17, 48, 3, 96, 3, True), (33, 16, 5, 32, 4, True)])
def test_one_launch_prologues(rt, abi, family, m, cols, blocks, kt, loop, extremes, order):
    """The element-wise operators in front of the one-launch kernel: half units of k, more than one 16-row piece,
    one and more 16-column pieces; infinities and NaN in the last rows and the last k of an iteration."""
    import numpy as np
    from attention_superoptimizer_amd import workloads as W
    from helpers import assert_f16_close, normal_f16
    from test_gpu_f16 import _graph_f16
    from test_gpu_launch_records import _kernel as launched
    k, n = kt * loop, cols * blocks
    acts, rows, cols_map = [W._inp([m, k])], (-1, -1, -1), (1, -1, -1)
    ops = [(f"tb_{family}_op", [(0, 0)]), ("tb_matmul_op", [(2, 0), (1, 0)])]
    if family == "silu_mul":
        acts.append(W._inp([m, k]))
        ops = [("tb_silu_op", [(0, 0)]), ("tb_mul_op", [(3, 0), (1, 0)]), ("tb_matmul_op", [(4, 0), (2, 0)])]
    na = len(acts)
    spec = acts + [W._inp([k, n], order),
                   {"op": "customized", "in": [[i, 0] for i in range(na + 1)],
                    "plan": W._plan((blocks, 1, 1), loop, [rows] * na + [cols_map], (1,) * na + (0,), cols_map, ops)}]
    # (one sign: no cancellation between iterations)
    ins = {i: abs(normal_f16(spec[i]["dims"], 0.1, 5 + i)) for i in range(na + 1)}
    if extremes:
        x, w = ins[0], ins[na]
        x[m - 1, kt - 1], x[m - 1, 0], x[16, -1], x[3, kt], x[0, 5] = np.inf, -np.inf, np.nan, 60000, -60000
        w[kt - 1, 1], w[-1, -1], w[kt, 4] = np.inf, np.nan, 50000
        if family == "silu_mul":
            ins[1][m - 2, -1], ins[1][m - 3, kt - 1] = np.inf, np.nan
    assert abi.mi355_set_option(7, 2) == 0
    try:
        got = _graph_f16(rt, spec, ins)[na + 1][0]
        pieces = cols // 16 * ((m + 15) // 16)
        assert launched() == (4, (blocks + 7) // 8 * 8 * pieces)  # the one-launch kernel's workgroups
    finally:
        assert abi.mi355_set_option(7, 0) == 0
    if extremes:
        assert abi.mi355_set_option(1, 1) == 0
        try:
            want = _graph_f16(rt, spec, ins)[na + 1][0]
        finally:
            assert abi.mi355_set_option(1, 0) == 0
        assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isposinf(got), np.isposinf(want))
        assert np.array_equal(np.isneginf(got), np.isneginf(want))
        ok = np.isfinite(want)
        assert ok.any() and not ok.all()
        assert_f16_close(got[ok], want[ok], what=family)
    else:
        from oracle import evaluate as orc
        assert_f16_close(got, orc.eval_graph(spec, "f16", ins, threads=8)[na + 1][0], what=family)


@pytest.mark.parametrize("order", [COL, ROW])
@pytest.mark.parametrize("m,blocks,kt,loop,col_groups,row_groups", [
    (8, 129, 64, 11, 8, 1), (16, 256, 64, 4, 8, 1), (9, 150, 128, 5, 8, 1),  # both weights in a workgroup, row-major
    (8, 130, 64, 40, 1, 1),   # and where strips leave no room for two workgroups on a compute unit
    (16, 129, 64, 33, 10, 10),  # results of both do not fit, one's do not either: ranges
    (8, 129, 64, 8, 8, 2), (8, 128, 64, 11, 8, 2), (16, 257, 64, 4, 8, 2),  # one weight in a workgroup
    (8, 65, 256, 16, 8, 2), (8, 40, 256, 16, 8, 6), (8, 63, 256, 32, 8, 16),  # whole for-loops, ranges in one round, in several
    (8, 64, 256, 16, 8, 4), (16, 32, 64, 31, 8, 8), (9, 32, 128, 28, 8, 14)])  # both weights, a range for every compute unit
def test_two_weights_in_a_workgroup(rt, ranges, m, blocks, kt, loop, col_groups, row_groups, order):
    """Which of its forms the streaming kernel takes for two weights (workgroups to a block), and their sums."""
    from attention_superoptimizer_amd import workloads as W
    from test_gpu_launch_records import _kernel as launched
    spec, _ = W.config5_gated_mlp(m=m, d=kt * loop, h=64 * blocks, grid1=blocks, F1=loop, grid2=kt * loop // 64, F2=blocks)
    spec = [op for i, op in enumerate(spec[:5]) if i != 3]
    _run(rt, spec, order, f"two weights {m} x {blocks}, {kt} x {loop}", std=0.05)
    assert launched()[1] == blocks * (col_groups if order == COL else row_groups)


@pytest.mark.parametrize("order", [COL, ROW])
@pytest.mark.parametrize("m,blocks,kt,loop,col_groups,row_groups", [
    (8, 129, 64, 45, 1, 1), (5, 200, 256, 16, 1, 1), (8, 129, 256, 16, 4, 1), (9, 129, 64, 13, 1, 1), (8, 128, 64, 33, 7, 7),
    (8, 40, 256, 32, 8, 6)])  # (row-major 256-k iterations: one round of workgroups)
def test_a_second_product_in_one_range(rt, ranges, m, blocks, kt, loop, col_groups, row_groups, order):
    """SiLU(a) * u in one range where its blocks are more than half of the compute units, up to 12 steps a
    wavefront (more of them from 192 blocks on)."""
    from attention_superoptimizer_amd import workloads as W
    from test_gpu_launch_records import _kernel as launched
    k, n, rows = kt * loop, 64 * blocks, (-1, -1, -1)
    spec = [W._inp([m, k]), W._inp([k, n], COL),
            {"op": "customized", "in": [[0, 0], [0, 0], [1, 0]],
             "plan": W._plan((blocks, 1, 1), loop, [rows, rows, (1, -1, -1)], (1, 1, 0), (1, -1, -1),
                             [("tb_silu_op", [(0, 0)]), ("tb_mul_op", [(3, 0), (1, 0)]), ("tb_matmul_op", [(4, 0), (2, 0)])])}]
    _run(rt, spec, order, f"second product {m} x {blocks}, {kt} x {loop}", std=0.1)
    assert launched()[1] == blocks * (col_groups if order == COL else row_groups)


@pytest.mark.parametrize("family,m,blocks,kt,loop,order,groups", [
    ("silu", 8, 5, 256, 40, COL, 50), ("lora", 4, 7, 64, 238, COL, 238), ("two", 4, 31, 64, 149, COL, 1178),
    ("plain", 4, 2, 256, 90, ROW, 46), ("plain", 4, 4, 256, 70, COL, 72),  # k for hundreds of iterations: ranges
    ("silu", 8, 5, 64, 8, COL, 32), ("lora", 4, 7, 64, 16, COL, 32), ("two", 4, 31, 64, 20, COL, 128),
    ("plain", 4, 2, 256, 12, ROW, 32), ("plain", 4, 4, 256, 16, COL, 32)])  # fewer: one launch
def test_the_rule_counts_the_chain_of_iterations(rt, family, m, blocks, kt, loop, order, groups):
    from attention_superoptimizer_amd import workloads as W
    from test_gpu_launch_records import _kernel as launched
    k, n, rows, cols = kt * loop, 64 * blocks, (-1, -1, -1), (1, -1, -1)
    if family == "lora":
        spec, _ = W.config4_lora(m=m, d=k, r=16, grid=blocks, F=loop)
        spec[1], spec[3] = W._inp([k, n], COL), W._inp([16, n], COL)
    elif family == "two":
        spec = [W._inp([m, k]), W._inp([k, n], COL), W._inp([k, n], COL),
                {"op": "customized", "in": [[0, 0], [1, 0], [2, 0]],
                 "plan": W._plan((blocks, 1, 1), loop, [rows, cols, cols], (1, 0, 0), cols,
                                 [("tb_matmul_op", [(0, 0), (1, 0)]), ("tb_matmul_op", [(0, 0), (2, 0)])])}]
    else:
        ops = [("tb_matmul_op", [(0, 0), (1, 0)])] if family == "plain" else [("tb_silu_op", [(0, 0)]), ("tb_matmul_op", [(2, 0), (1, 0)])]
        spec = [W._inp([m, k]), W._inp([k, n], COL),
                {"op": "customized", "in": [[0, 0], [1, 0]], "plan": W._plan((blocks, 1, 1), loop, [rows, cols], (1, 0), cols, ops)}]
    _run(rt, spec, order, f"{family} {m} x {blocks}, {kt} x {loop}", std=0.03)
    assert launched()[1] == groups
