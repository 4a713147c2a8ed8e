"""The attention kernel for tiles of any size against the fp16 oracle: query tiles around the edges
of a 16-row group and of a wavefront's row groups, key tiles of an odd and an even number of
16-key blocks (one block, a lone last block, more than one chunk of registers), fewer and more
iterations than lanes, both forms, both storage orders, row tiles that join into one tall tile."""
import pytest

from helpers import assert_f16_close, normal_f16
from oracle import evaluate as orc
from test_gpu_f16 import KERNEL_ATTENTION, _graph_f16, _last_kernels

pytestmark = pytest.mark.gpu
ROW, COL = "DmemRowMajor", "DmemColumnMajor"


def _inputs(spec, std):
    ins = {i: normal_f16(op["dims"], std, 11 + i) for i, op in enumerate(spec) if op["op"] == "input"}
    ins[2] = abs(ins[2])  # (no cancellation between iterations)
    return ins


def _run(rt, spec, what, std=0.125):
    ins = _inputs(spec, std)
    got = _graph_f16(rt, spec, ins)
    want = orc.eval_graph(spec, "f16", ins, threads=8)
    for i, op in enumerate(spec):
        if op["op"] == "customized":
            for j, w in enumerate(want[i]):
                assert_f16_close(got[i][j], w, what=f"{what} op {i} out {j}")
    assert _last_kernels[0] == KERNEL_ATTENTION, what


# rows, key tile, for-loop
SHAPES = [(1, 48, 5), (15, 16, 1), (17, 80, 3), (33, 64, 9), (64, 48, 2), (65, 112, 4), (130, 32, 13)]


@pytest.mark.parametrize("order", [COL, ROW])
@pytest.mark.parametrize("rows,keys,loop", SHAPES)
def test_both_forms(rt, rows, keys, loop, order):
    from attention_superoptimizer_amd import workloads as W
    for make in (W.config2_gqa_decode, W.gqa_inc_decode):  # with the division, and without it
        spec, _ = make(groups=3, rows=rows, seq=keys * 2 * loop, kv_blocks=2, F=loop)
        for i in (1, 2):
            spec[i]["layout"] = order
        _run(rt, spec, f"{make.__name__} {rows} rows {keys} keys x {loop} {order}")


@pytest.mark.parametrize("order", [COL, ROW])
@pytest.mark.parametrize("hd,row_tile,blocks,keys,loop", [
    (64, 80, 13, 80, 13), (64, 48, 40, 144, 3), (128, 48, 3, 32, 5), (128, 80, 9, 112, 6), (128, 24, 20, 80, 2)])
def test_prefill_row_tiles_join(rt, hd, row_tile, blocks, keys, loop, order):
    from attention_superoptimizer_amd import workloads as W
    heads = 12 if row_tile == 80 and hd == 64 else 3
    rows, seq = row_tile * blocks, keys * loop
    spec = [W._inp([heads, rows, hd]), W._inp([heads, hd, seq], order), W._inp([heads, seq, hd], order),
            {"op": "customized", "in": [[0, 0], [1, 0], [2, 0]],
             "plan": W._plan((heads, 1, blocks), loop, [(0, -1, 1), (0, 2, -1), (0, 1, -1)], (-1, 2, 1), (0, 2, 1),
                             W.ATT_OPS, dimx=hd)}]
    _run(rt, spec, f"prefill {hd} {row_tile} x {blocks}, {keys} x {loop} {order}")
