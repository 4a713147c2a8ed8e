"""The fused fingerprint attention kernel and the one-pass exp / row sum / division, bit for bit."""
import ctypes

import numpy as np
import pytest

from attention_superoptimizer_amd import _native as N
from attention_superoptimizer_amd import workloads as W
from helpers import FP_PQ, uniform_fp
from oracle import evaluate as orc

pytestmark = pytest.mark.gpu

SUMS = [("tb_matmul_op", [(0, 0), (1, 0)]), ("tb_exp_op", [(3, 0)]), ("tb_matmul_op", [(4, 0), (2, 0)]),
        ("tb_reduction_2_op", [(4, 0)])]
DIVIDED = [("tb_matmul_op", [(0, 0), (1, 0)]), ("tb_exp_op", [(3, 0)]), ("tb_reduction_2_op", [(4, 0)]),
           ("tb_div_op", [(4, 0), (5, 0)]), ("tb_matmul_op", [(6, 0), (2, 0)])]
BY_SCORES = [("tb_matmul_op", [(0, 0), (1, 0)]), ("tb_reduction_2_op", [(3, 0)]), ("tb_exp_op", [(3, 0)]),
             ("tb_div_op", [(5, 0), (4, 0)]), ("tb_matmul_op", [(6, 0), (2, 0)])]


def _spec(form, b, m, row_blocks, n, F, kv_blocks, d, dv):
    keys = n * F * kv_blocks
    ops = {"sums": SUMS, "divided": DIVIDED, "scores": BY_SCORES}[form]
    outs = [(0, 2, 1)]
    q, k, v = [b, m * row_blocks, d], [b, d, keys], [b, keys, dv]
    plan = W._plan((b, kv_blocks, row_blocks), F, [(0, -1, 1), (0, 2, -1), (0, 1, -1)], (-1, 2, 1), outs[0], ops, dimx=dv)
    return [{"op": "input", "dims": q}, {"op": "input", "dims": k}, {"op": "input", "dims": v},
            {"op": "customized", "in": [[0, 0], [1, 0], [2, 0]], "plan": plan}]


@pytest.mark.parametrize("form", ["sums", "divided", "scores"])
@pytest.mark.parametrize("b,m,row_blocks,n,F,kv_blocks,d,dv", [
    (1, 16, 1, 64, 1, 1, 64, 64),
    (2, 1, 3, 16, 2, 2, 64, 64),      # fewer rows than a row group, fewer keys than a chunk
    (1, 24, 2, 48, 3, 2, 64, 64),     # two row groups, the second short
    (1, 48, 1, 208, 1, 1, 64, 64),    # four chunks, the last one short
    (3, 16, 1, 512, 2, 1, 64, 64),    # keys shared by four wavefronts
    (1, 130, 1, 64, 2, 1, 64, 64),    # more rows than a workgroup has
    (1, 20, 1, 80, 1, 1, 16, 32),     # short rows of K and V
])
def test_fused_fingerprint_attention(rt, abi, form, b, m, row_blocks, n, F, kv_blocks, d, dv):
    spec = _spec(form, b, m, row_blocks, n, F, kv_blocks, d, dv)
    for extreme in (False, True):
        ins = {i: np.full(spec[i]["dims"], FP_PQ - 1, np.uint16) if extreme else uniform_fp(spec[i]["dims"], 7 + i) for i in range(3)}
        g, vals = rt.build_from_spec(spec)
        try:
            for i, a in ins.items():
                vals[i][0].write_fingerprint(a)
            g.fingerprint(3)
            info = N.Mi355LaunchInfo()
            abi.mi355_last_launch(ctypes.byref(info))
            assert info.kernel_id == 7
            got = [t.read_fingerprint() for t in vals[3]]
        finally:
            g.close()
        for x, y in zip(got, orc.eval_graph(spec, "fp", ins)[3]):
            np.testing.assert_array_equal(x, y)


@pytest.mark.parametrize("form", ["sums", "divided", "scores"])
def test_fused_fingerprint_attention_of_any_16_bit_values(rt, form):
    spec = _spec(form, 4, 64, 2, 64, 2, 2, 64, 64)
    ins = {i: np.random.default_rng(i).permutation(np.resize(np.arange(65536, dtype=np.uint16), int(np.prod(spec[i]["dims"]))))
           .reshape(spec[i]["dims"]) for i in range(3)}
    g, vals = rt.build_from_spec(spec)
    try:
        for i, a in ins.items():
            vals[i][0].write_fingerprint(a)
        g.fingerprint(3)
        got = [t.read_fingerprint() for t in vals[3]]
    finally:
        g.close()
    for x, y in zip(got, orc.eval_graph(spec, "fp", {i: a % FP_PQ for i, a in ins.items()})[3]):
        np.testing.assert_array_equal(x, y)


@pytest.mark.parametrize("form", ["sums", "divided", "scores"])
def test_fused_fingerprint_attention_in_a_batch(rt, abi, form):
    specs = [_spec(form, 2, 16, 2, 64, 2, 2, 64, 64), _spec(form, 2, 32, 1, 128, 1, 2, 64, 64)]
    graphs = [rt.build_from_spec(s) for s in specs]
    try:
        for (g, _), s in zip(graphs, specs):
            verdicts, _ = rt.verify_batch([g], g, 5)
            assert verdicts == [True]
            want = orc.eval_graph(s, "fp", {i: graphs_input(s, i, 5) for i in range(3)})[3]
            for t, w in zip(graphs[specs.index(s)][1][3], want):
                np.testing.assert_array_equal(t.read_fingerprint(), w)
    finally:
        for g, _ in reversed(graphs):
            g.close()


def graphs_input(spec, i, seed):
    return uniform_fp(spec[i]["dims"], seed ^ (i << 40))


@pytest.mark.parametrize("b,m,n", [(1, 1, 1), (2, 3, 7), (1, 5, 2047), (1, 5, 4097), (2, 600, 513), (1, 1025, 4096), (1, 2, 20001)])
def test_fingerprint_softmax_rows(rt, abi, b, m, n):
    spec = [{"op": "input", "dims": [b, m, n]}, {"op": "exp", "in": [[0, 0]]},
            {"op": "reduction", "in": [[1, 0]], "dim": 2, "size": 1}, {"op": "div", "in": [[1, 0], [2, 0]]}]
    g, vals = rt.build_from_spec(spec)
    try:
        g.fingerprint_seeded(9)
        want = orc.eval_graph(spec, "fp", {0: uniform_fp([b, m, n], 9)})
        for t, w in zip(vals, want):
            np.testing.assert_array_equal(t[0].read_fingerprint(), w[0])
    finally:
        g.close()
