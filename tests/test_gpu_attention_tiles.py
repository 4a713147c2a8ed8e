"""The attention kernel for tiles of any size against the fp16 oracle: query tiles around the edges
of a 16-row group and of a wavefront's row groups, key tiles of an odd and an even number of
16-key blocks (one block, a lone last block, more than one chunk of registers), fewer and more
iterations than lanes, both forms, both storage orders, row tiles that join into one tall tile."""
import numpy as np
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
SHAPES = [(1, 48, 5), (15, 16, 1), (17, 80, 3), (33, 64, 9), (64, 48, 2), (65, 112, 4), (130, 32, 13),
          (7, 80, 1), (5, 32, 9), (12, 16, 17), (3, 112, 9)]  # one to six pairs of key blocks a wavefront, odd and even


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


@pytest.mark.parametrize("order", [COL, ROW])
@pytest.mark.parametrize("rows,keys,loop", [(5, 16, 1), (5, 48, 3), (40, 80, 2), (33, 112, 9)])
def test_keys_of_other_tiles_do_not_matter(rt, rows, keys, loop, order):
    """The keys around a thread block's own are infinities and NaN: a lone last block of a tile is read as
    half of a pair, and a block of a wavefront ahead of its turn."""
    from attention_superoptimizer_amd import workloads as W
    for make in (W.config2_gqa_decode, W.gqa_inc_decode):
        spec, _ = make(groups=2, rows=rows, seq=keys * loop * 3, kv_blocks=3, F=loop)
        for i in (1, 2):
            spec[i]["layout"] = order
        ins = _inputs(spec, 0.125)
        clean = _graph_f16(rt, spec, ins)[3]
        mine = slice(keys * loop, 2 * keys * loop)  # the second of the three thread blocks that share a query tile
        for i, axis in ((1, 2), (2, 1)):
            odd = np.full_like(ins[i], np.nan)
            odd[::2] = np.inf
            at = [slice(None)] * 3
            at[axis] = mine
            odd[tuple(at)] = ins[i][tuple(at)]
            ins[i] = odd
        got = _graph_f16(rt, spec, ins)[3]
        assert _last_kernels[0] == KERNEL_ATTENTION
        for g, w in zip(got, clean):
            third = g.shape[-1] // 3
            np.testing.assert_array_equal(g[..., third:2 * third], w[..., third:2 * third])


def _tile_values(rt, make, groups, keys, order, scores, v):
    """A plan's first results for one iteration of `keys` keys: rows of one-hot queries, so that the scores
    are the keys' values themselves."""
    spec, _ = make(groups=groups, rows=64, seq=keys, kv_blocks=1, F=1)
    for i in (1, 2):
        spec[i]["layout"] = order
    q = np.broadcast_to(np.eye(64, dtype=np.float16), (groups, 64, 64))
    got = _graph_f16(rt, spec, {0: q, 1: scores, 2: v})
    assert _last_kernels[0] == KERNEL_ATTENTION
    return got[3]


@pytest.mark.parametrize("order", [COL, ROW])
@pytest.mark.parametrize("keys", [16, 48])
@pytest.mark.parametrize("peaked", [False, True], ids=["even", "peaked"])
def test_division_is_the_quotient(rt, keys, order, peaked):
    """P = E / sum to the bit, with E of a few units, and with sums of 6 and 12 next to which the other keys
    vanish: their quotients are subnormal numbers, many in the middle of two.  E and the sums come from the
    form without the division, the values of V show P one by one; E is of a range in which any order of
    adding gives the same fp16 sum."""
    from attention_superoptimizer_amd import workloads as W
    groups = 64
    rng = np.random.default_rng(keys)
    scores = rng.uniform(*((-16.6, -10.4) if peaked else (-2.7, 2.0)), (groups, 64, keys)).astype(np.float16)
    if peaked:
        scores[::2, :, :6] = scores[1::2, :, :12] = 0
    v = np.zeros((groups, keys, 64), np.float16)
    v[:, np.arange(keys), np.arange(keys)] = 1
    e, sums = _tile_values(rt, W.gqa_inc_decode, groups, keys, order, scores, v)
    p = _tile_values(rt, W.config2_gqa_decode, groups, keys, order, scores, v)[0]
    e, sums = e.reshape(groups, 64, 64)[:, :, :keys].astype(np.float32), sums.reshape(groups, 64, -1)[:, :, :1].astype(np.float32)
    assert np.array_equal(e.astype(np.float64).sum(2, keepdims=True).astype(np.float16).astype(np.float32), sums)
    assert not peaked or set(sums.ravel()) == {6, 12}
    np.testing.assert_array_equal(p.reshape(groups, 64, 64)[:, :, :keys], (e / sums).astype(np.float16))


@pytest.mark.parametrize("order", [COL, ROW])
def test_division_of_sums_out_of_range(rt, abi, order):
    """Scores whose exponentials overflow or vanish, infinities and NaN: what the interpreter's statements
    give, number for number."""
    from attention_superoptimizer_amd import workloads as W
    groups, keys = 3, 48
    rng = np.random.default_rng(9)
    scores = rng.uniform(-1, 1, (groups, 64, keys)).astype(np.float16)
    scores[0, 0] = -30          # every exponential and the sum are zero: no number
    scores[0, 1] = 9            # the sum is infinite, no exponential is: zeros
    scores[0, 2, 5] = 12        # one exponential and the sum are infinite
    scores[0, 3] = -16          # the smallest numbers
    scores[1, 0, 7] = 11.09     # close to the largest
    v = np.broadcast_to(np.eye(keys, 64, dtype=np.float16), (groups, keys, 64))
    for make in (W.gqa_inc_decode, W.config2_gqa_decode):
        fused = _tile_values(rt, make, groups, keys, order, scores, v)
        assert abi.mi355_set_option(1, 1) == 0
        try:
            _last_kernels[:] = []
            spec, _ = make(groups=groups, rows=64, seq=keys, kv_blocks=1, F=1)
            for i in (1, 2):
                spec[i]["layout"] = order
            want = _graph_f16(rt, spec, {0: np.broadcast_to(np.eye(64, dtype=np.float16), (groups, 64, 64)), 1: scores, 2: v})[3]
        finally:
            assert abi.mi355_set_option(1, 0) == 0
        for f, w in zip(fused, want):
            assert np.array_equal(np.isnan(f), np.isnan(w)) and np.array_equal(np.isposinf(f), np.isposinf(w))
            ok = np.isfinite(w)
            assert_f16_close(f[ok], w[ok], what=make.__name__)


@pytest.mark.parametrize("order", [COL, ROW])
@pytest.mark.parametrize("rows,keys", [(8, 64), (3, 48)])
def test_every_block_of_a_long_cache_runs_once(rt, rows, keys, order):
    """More than 128 MB of keys and values: blocks then run in launch order, key blocks before groups.  Every
    score is zero and every value of a block one number of its own, so that sums are exact up to the fp16
    additions of the iterations, which numpy does as well."""
    from attention_superoptimizer_amd import workloads as W
    groups, kv_blocks = 16, 64
    loop = 1 + (128 << 20) // (groups * kv_blocks * keys * 64 * 4)
    seq = keys * loop * kv_blocks
    spec, _ = W.gqa_inc_decode(groups=groups, rows=rows, seq=seq, kv_blocks=kv_blocks, F=loop)
    for i in (1, 2):
        spec[i]["layout"] = order
    ids = (1 + np.arange(groups * kv_blocks).reshape(groups, kv_blocks) / 1024).astype(np.float16)
    v = np.broadcast_to(np.repeat(ids, keys * loop, 1)[:, :, None], (groups, seq, 64))
    o, r = _graph_f16(rt, spec[:4], {0: np.zeros((groups, rows, 64), np.float16), 1: normal_f16([groups, 64, seq], 1.0, 3), 2: v})[3]
    assert _last_kernels[0] == KERNEL_ATTENTION
    tile = (ids.astype(np.float64) * keys).astype(np.float16)
    want, sums = np.zeros_like(tile), np.float16(0)
    for _ in range(loop):
        want, sums = want + tile, sums + np.float16(keys)
    np.testing.assert_array_equal(r, np.full_like(r, sums))
    np.testing.assert_array_equal(o.reshape(groups, rows, kv_blocks, 64), np.broadcast_to(want[:, None, :, None], (groups, rows, kv_blocks, 64)))
