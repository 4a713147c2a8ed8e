"""Performance cases of the framework: what a program that uses it runs, through `KNGraph`.

Three kinds of program use the framework, and every case belongs to one of them:

* one that RUNS mugraphs in fp16: it builds a graph once, keeps its tensors in device memory and
  calls `execute_all` for every step (decode and prefill attention, fused matmul, LoRA, gated MLP);
* one that runs the UN-FUSED graph of the same computation, the thing a mugraph is compared with
  (kernel-level matmuls, element-wise operators and reductions, any sizes);
* a SEARCH: it proves candidates equal to a graph by fingerprints in Z_25651, one candidate at a
  time (`fingerprint_seeded`, `has_same_fingerprint`) or a batch at a time (`verify_batch_*`).

Sizes are those of `workloads.py` and `candidates.py` and the ranges around them: decode steps
from one query row up, key tiles and row tiles that are multiples of 16 and ones that are not,
both storage orders of keys, values and weights.
"""
import math
import random

import numpy as np
import torch

from attention_superoptimizer_amd import graph as G
from attention_superoptimizer_amd import workloads as W

ROW, COL = "DmemRowMajor", "DmemColumnMajor"
LAYOUTS = {"row": ROW, "col": COL}
KN_INPUT_OP = 1001


# ---------------------------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------------------------
def listed():
    return [
        # One decode step as one operator, softmax included: the benchmark's headline configuration
        # and the smallest call here -- a serving loop repeats it per layer and token.
        {"name": "decode_one_op", "kind": "decode", "groups": 2, "rows": 256, "key_tile": 64, "kv_blocks": 16,
         "loop": 4, "order": "col"},
        # Split-KV decode against a long cache: 8 query rows per kv-head group, 16,384 keys, more
        # bytes of K and V than any cache holds.  The bandwidth-bound end of decoding.
        {"name": "decode_long_cache", "kind": "split_kv", "groups": 64, "rows": 8, "key_tile": 64, "kv_blocks": 16,
         "loop": 16, "order": "col"},
        # Split-KV decode at sizes nobody tuned for: 5 groups, 12 query rows, key tiles of 48, keys
        # and values row-major (a cache written by another program).
        {"name": "decode_odd_tiles", "kind": "split_kv", "groups": 5, "rows": 12, "key_tile": 48, "kv_blocks": 12,
         "loop": 5, "order": "row"},
        # Prefill of 32 heads x 2048 tokens at head size 128: the largest attention configuration.
        {"name": "prefill_2048", "kind": "prefill", "heads": 32, "row_tile": 128, "row_blocks": 16, "head": 128,
         "key_tile": 64, "loop": 32, "order": "col"},
        # Prefill of a prompt whose length is not a power of two: 12 heads x 1040 tokens, tiles of 80.
        {"name": "prefill_1040", "kind": "prefill", "heads": 12, "row_tile": 80, "row_blocks": 13, "head": 64,
         "key_tile": 80, "loop": 13, "order": "col"},
        # A fused matmul operator of a few MB (64 x 1024 x 1024): launch latency counts.
        {"name": "matmul_op", "kind": "matmul_op", "m": 64, "col_tile": 64, "col_blocks": 16, "k_tile": 64,
         "loop": 16, "order": "col"},
        # LoRA linear layer of a decode step: 16 tokens, 4096 x 4096, rank 16.
        {"name": "lora_4096", "kind": "lora", "m": 16, "rank": 16, "col_tile": 64, "col_blocks": 64, "k_tile": 256,
         "loop": 16, "order": "col"},
        # Gated MLP of a decode step: 8 tokens, 4096 x 14336, two operators, 353 MB of weights.
        {"name": "gated_mlp_14336", "kind": "gated_mlp", "m": 8, "d_blocks": 64, "h_blocks": 224, "k_tile": 256,
         "order": "col"},
        # The un-fused attention graph on ragged sizes: what a search starts from and times first.
        {"name": "unfused_attention", "kind": "unfused_attention", "heads": 8, "rows": 500, "keys": 1000, "head": 64,
         "order": "col"},
        # The un-fused gated MLP over a prompt of 300 tokens with weights row-major and a hidden size
        # that is no power of two: kernel-level GEMMs and element-wise operators.
        {"name": "unfused_mlp", "kind": "unfused_mlp", "m": 300, "d": 2048, "h": 5504, "order": "row"},
        # One candidate proved equal to its un-fused graph: both fingerprinted, outputs compared.
        {"name": "equivalence", "kind": "equivalence", "heads": 32, "rows": 256, "row_tile": 64, "key_tile": 64,
         "kv_blocks": 4, "loop": 4, "head": 64},
        # One step of a search: 48 candidates are built from their plans, verified as a batch with
        # their reference graph, and dropped.
        {"name": "search_step", "kind": "search", "family": "mlp", "m": 64, "k": 512, "h": 512, "n": 512, "candidates": 48,
         "built": False},
    ]


def _near(rng, lo, hi):
    """A whole number between lo and hi, spread over the logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _tiles_fit(rows, key_tile, head):
    """Whether the tiles of an attention operator fit a thread block's LDS on every route."""
    return 2 * (3 * rows * head + 2 * key_tile * head + 2 * rows * key_tile) <= 120 * 1024


def _draw_decode(rng):
    while True:
        c = {"kind": "decode", "groups": _near(rng, 1, 16), "rows": rng.choice([rng.randint(1, 64), 16 * rng.randint(1, 16)]),
             "key_tile": rng.choice([16, 32, 48, 64, 64, 80, 96, 128]), "kv_blocks": _near(rng, 2, 32),
             "loop": rng.randint(1, 8), "order": rng.choice(["col", "col", "row"])}
        if _tiles_fit(c["rows"], c["key_tile"], 64):
            return c


def _draw_split_kv(rng):
    while True:
        c = {"kind": "split_kv", "groups": _near(rng, 1, 64), "rows": rng.choice([1, rng.randint(1, 64), 8, 16]),
             "key_tile": rng.choice([16, 32, 48, 64, 64, 80, 128]), "kv_blocks": _near(rng, 2, 32),
             "loop": rng.randint(1, 16), "order": rng.choice(["col", "col", "row"])}
        keys = c["key_tile"] * c["kv_blocks"] * c["loop"]  # (their exponentials' sum has to stay an fp16 number)
        if keys <= 32768 and c["groups"] * keys <= 64 * 16384 and _tiles_fit(c["rows"], c["key_tile"], 64):
            return c


def _draw_prefill(rng):
    while True:
        c = {"kind": "prefill", "heads": _near(rng, 2, 40), "row_tile": rng.choice([32, 48, 64, 80, 96, 128, 128]),
             "row_blocks": _near(rng, 2, 32), "head": rng.choice([64, 64, 128]),
             "key_tile": rng.choice([32, 48, 64, 64, 80, 128]), "order": rng.choice(["col", "col", "row"])}
        tokens = c["row_tile"] * c["row_blocks"]
        c["loop"] = tokens // c["key_tile"]  # self-attention, the last keys short of a whole tile left out
        work = c["heads"] * tokens * c["loop"] * c["key_tile"] * c["head"]
        if c["loop"] >= 1 and work <= 32 * 2048 * 2048 * 128 / 4 and _tiles_fit(c["row_tile"], c["key_tile"], c["head"]):
            return c


def _draw_matmul_op(rng):
    return {"kind": "matmul_op", "m": rng.choice([rng.randint(1, 64), 16, 32, 64]), "col_tile": rng.choice([32, 48, 64, 64, 128]),
            "col_blocks": _near(rng, 4, 128), "k_tile": rng.choice([32, 64, 96, 128, 256]), "loop": _near(rng, 2, 32),
            "order": rng.choice(["col", "col", "row"])}


def _draw_lora(rng):
    return {"kind": "lora", "m": rng.choice([16, rng.randint(1, 32)]), "rank": rng.choice([8, 16, 16, 32]), "col_tile": 64,
            "col_blocks": _near(rng, 8, 64), "k_tile": rng.choice([64, 128, 256]), "loop": _near(rng, 2, 16),
            "order": rng.choice(["col", "col", "row"])}


def _draw_gated_mlp(rng):
    return {"kind": "gated_mlp", "m": rng.choice([8, 16, rng.randint(1, 16)]), "d_blocks": _near(rng, 8, 64),
            "h_blocks": _near(rng, 16, 224), "k_tile": rng.choice([64, 128, 256]), "order": rng.choice(["col", "col", "row"])}


def _draw_unfused_attention(rng):
    while True:
        c = {"kind": "unfused_attention", "heads": _near(rng, 1, 32), "rows": _near(rng, 1, 2048), "keys": _near(rng, 64, 4096),
             "head": rng.choice([64, 128]), "order": rng.choice(["col", "col", "row"])}
        if c["heads"] * c["rows"] * c["keys"] <= 32 * 1024 * 1024:
            return c


def _draw_unfused_mlp(rng):
    return {"kind": "unfused_mlp", "m": _near(rng, 1, 1024), "d": _near(rng, 256, 2048), "h": _near(rng, 512, 5504),
            "order": rng.choice(["col", "row"])}


def _draw_equivalence(rng):
    return {"kind": "equivalence", "heads": _near(rng, 1, 32), "rows": 0, "row_tile": rng.choice([16, 24, 32, 48, 64]),
            "key_tile": rng.choice([32, 48, 64, 64]), "kv_blocks": _near(rng, 2, 8), "loop": rng.randint(1, 4), "head": 64,
            "row_blocks": rng.randint(1, 4)}


def _draw_search(rng):
    p = lambda lo, hi: 2 ** rng.randint(int(math.log2(lo)), int(math.log2(hi)))  # noqa: E731
    return {"kind": "search", "family": rng.choice(["matmul_add", "mlp", "attention", "row_softmax"]), "m": p(64, 256),
            "k": p(64, 512), "h": p(64, 512), "n": p(64, 512), "candidates": rng.randint(1, 48), "built": rng.random() < 0.5}


_DRAW = [_draw_decode, _draw_split_kv, _draw_prefill, _draw_matmul_op, _draw_lora, _draw_gated_mlp,
         _draw_unfused_attention, _draw_unfused_mlp, _draw_equivalence, _draw_search]


def draw(rng):
    c = rng.choice(_DRAW)(rng)
    if c["kind"] == "equivalence":
        c["rows"] = c["row_tile"] * c.pop("row_blocks")
    return c


# ---------------------------------------------------------------------------------------------
# graphs of a case
# ---------------------------------------------------------------------------------------------
def _in_order(spec, order):
    """The weight-side inputs (declared column-major by the plans) in the storage order asked for."""
    return [dict(op, layout=LAYOUTS[order]) if op["op"] == "input" and op["layout"] == COL else op for op in spec]


def _gated_mlp(c):
    d, h, kt = 64 * c["d_blocks"], 64 * c["h_blocks"], c["k_tile"]
    kt1, kt2 = math.gcd(d, kt), math.gcd(h, kt)
    return W.config5_gated_mlp(m=c["m"], d=d, h=h, grid1=c["h_blocks"], F1=d // kt1, grid2=c["d_blocks"], F2=h // kt2)


def _specs(c):
    """(mugraph, un-fused graph) of a case as graph specs."""
    k = c["kind"]
    if k == "decode":
        g, _ = W.config2_gqa_decode(c["groups"], c["rows"], c["key_tile"] * c["kv_blocks"] * c["loop"], c["kv_blocks"], c["loop"])
        return _in_order(g, c["order"]), None
    if k == "split_kv":
        g, r = W.gqa_inc_decode(c["groups"], c["rows"], c["key_tile"] * c["kv_blocks"] * c["loop"], c["kv_blocks"], c["loop"])
        return _in_order(g, c["order"]), r
    if k == "prefill":
        tokens, keys, hd = c["row_tile"] * c["row_blocks"], c["key_tile"] * c["loop"], c["head"]
        q, kk, v = [c["heads"], tokens, hd], [c["heads"], hd, keys], [c["heads"], keys, hd]
        g = [W._inp(q), W._inp(kk, COL), W._inp(v, COL),
             {"op": "customized", "in": [[0, 0], [1, 0], [2, 0]],
              "plan": W._plan((c["heads"], 1, c["row_blocks"]), c["loop"], [(0, -1, 1), (0, 2, -1), (0, 1, -1)], (-1, 2, 1),
                              (0, 2, 1), W.ATT_OPS, dimx=hd)},
             {"op": "customized", "in": [[3, 0], [3, 1]],
              "plan": W._plan((c["heads"], tokens // 16, 1), 1, [(0, 1, -1), (0, 1, -1)], (-1, -1), (0, 1, -1),
                              W.COMBINE_OPS, dimx=hd)}]
        return _in_order(g, c["order"]), None
    if k == "matmul_op":
        g, r = W.tiled_matmul(c["m"], c["col_tile"] * c["col_blocks"], c["k_tile"] * c["loop"], (c["col_blocks"], 1, 1), c["loop"],
                              (-1, -1, -1), (1, -1, -1), (1, -1, -1))
        return _in_order(g, c["order"]), r
    if k == "lora":
        d, n, r, kt = c["k_tile"] * c["loop"], c["col_tile"] * c["col_blocks"], c["rank"], c["k_tile"]
        g, _ = W.config4_lora(m=c["m"], d=d, r=r, grid=c["col_blocks"], F=c["loop"])
        g[1], g[3] = W._inp([d, n], COL), W._inp([r, n], COL)  # as wide as the case says
        return _in_order(g, c["order"]), None
    if k == "gated_mlp":
        return _in_order(_gated_mlp(c)[0], c["order"]), None
    if k == "unfused_attention":
        b, m, s, hd = c["heads"], c["rows"], c["keys"], c["head"]
        return _in_order(W.attention_reference([b, m, hd], [b, hd, s], [b, s, hd]), c["order"]), None
    if k == "unfused_mlp":
        m, d, h = c["m"], c["d"], c["h"]
        return _in_order([
            W._inp([m, d]), W._inp([d, h], COL), W._inp([d, h], COL), W._inp([h, d], COL),
            {"op": "matmul", "in": [[0, 0], [1, 0]]}, {"op": "silu", "in": [[4, 0]]},
            {"op": "matmul", "in": [[0, 0], [2, 0]]}, {"op": "mul", "in": [[5, 0], [6, 0]]},
            {"op": "matmul", "in": [[7, 0], [3, 0]]}], c["order"]), None
    if k == "equivalence":
        b, m, hd, s = c["heads"], c["rows"], c["head"], c["key_tile"] * c["kv_blocks"] * c["loop"]
        q, kk, v = [b, m, hd], [b, hd, s], [b, s, hd]
        g = W.attention_two_stage(q, kk, v, (0, -1, 1), (0, 2, 1), (b, c["kv_blocks"], m // c["row_tile"]), c["loop"],
                                  (0, 1, -1), (b, m // 8, 1))
        return g, W.attention_reference(q, kk, v)
    raise ValueError(k)


def _matmul_plans(rng, m, n, k, unary=None):
    """Operators of one [m, k] . [k, n] matmul as a search tiles it: rows over grid y, columns over
    grid x, k over the for-loop, every tile a power of two."""
    mt = rng.choice([t for t in (16, 32, 64, 128) if t <= m])
    nt = rng.choice([t for t in (32, 64, 128) if t <= n])
    kt = rng.choice([t for t in (32, 64, 128) if t <= k])
    gx, gy = n // nt, m // mt
    ops = [("tb_matmul_op", [(0, 0), (1, 0)])]
    if unary == "before":
        ops = [("tb_exp_op", [(0, 0)]), ("tb_matmul_op", [(2, 0), (1, 0)])]
    elif unary == "after":
        ops.append(("tb_exp_op", [(2, 0)]))
    return W._plan((gx, gy, 1), k // kt, [(-1, 0 if gy > 1 else -1, -1), (1 if gx > 1 else -1, -1, -1)], (1, 0),
                   (1 if gx > 1 else -1, 0 if gy > 1 else -1, -1), ops)


def _search_specs(c, seed):
    """The reference graph of a search and its candidates' specs; about a quarter of the candidates
    compute something else."""
    rng = random.Random(seed)
    m, k, h, n = c["m"], c["k"], c["h"], c["n"]
    if c["family"] == "attention":
        b, s = max(1, h // 64), n
        q, kk, v = [b, m, 64], [b, 64, s], [b, s, 64]
        ref = W.attention_reference(q, kk, v)

        def candidate(wrong):
            mq = rng.choice([t for t in (16, 32, 64) if t <= m])
            if s > 256:
                mq = min(mq, 16)
            qi, ki = ((0 if b > 1 else -1), -1, (1 if m > mq else -1)), ((0 if b > 1 else -1), -1, -1)
            ops = [("tb_matmul_op", [(0, 0), (1, 0)]), ("tb_exp_op", [(3, 0)]), ("tb_reduction_2_op", [(4, 0)]),
                   ("tb_div_op", [(4, 0), (5, 0)]), ("tb_matmul_op", [(6, 0), (2, 0)])]
            if wrong:  # the row sums are taken before the exponential
                ops[1:4] = [("tb_reduction_2_op", [(3, 0)]), ("tb_exp_op", [(3, 0)]), ("tb_div_op", [(5, 0), (4, 0)])]
            return ref[:3] + [{"op": "customized", "in": [[0, 0], [1, 0], [2, 0]],
                               "plan": W._plan((b, 1, m // mq), 1, [qi, ki, ki], (-1, -1, -1), qi, ops)}]
    elif c["family"] == "matmul_add":
        ref = [W._inp([m, k]), W._inp([k, n], COL), W._inp([m, n]), {"op": "matmul", "in": [[0, 0], [1, 0]]},
               {"op": "add", "in": [[3, 0], [2, 0]]}]

        def candidate(wrong):
            return ref[:3] + [{"op": "customized", "in": [[0, 0], [1, 0]], "plan": _matmul_plans(rng, m, n, k, "after" if wrong else None)},
                              {"op": "add", "in": [[3, 0], [2, 0]]}]
    elif c["family"] == "mlp":
        m = min(m, 128)
        ref = [W._inp([m, k]), W._inp([k, h], COL), W._inp([h, n], COL), {"op": "matmul", "in": [[0, 0], [1, 0]]},
               {"op": "exp", "in": [[3, 0]]}, {"op": "matmul", "in": [[4, 0], [2, 0]]}]

        def candidate(wrong):
            first = {"op": "matmul", "in": [[0, 0], [1, 0]]}
            if rng.random() < 0.5:
                first = {"op": "customized", "in": [[0, 0], [1, 0]], "plan": _matmul_plans(rng, m, h, k)}
            return ref[:3] + [first, {"op": "customized", "in": [[3, 0], [2, 0]],
                                      "plan": _matmul_plans(rng, m, n, h, None if wrong else "before")}]
    else:  # row softmax
        ref = [W._inp([m, k]), W._inp([k, n], COL), {"op": "matmul", "in": [[0, 0], [1, 0]]}, {"op": "exp", "in": [[2, 0]]},
               {"op": "reduction", "in": [[3, 0]], "dim": 1, "size": 1}, {"op": "div", "in": [[3, 0], [4, 0]]}]

        def candidate(wrong):
            first = {"op": "matmul", "in": [[0, 0], [1, 0]]}
            if rng.random() < 0.5:
                first = {"op": "customized", "in": [[0, 0], [1, 0]], "plan": _matmul_plans(rng, m, n, k)}
            mt = rng.choice([16, 32])
            ops = [("tb_exp_op", [(0, 0)]), ("tb_reduction_1_op", [(1, 0)]), ("tb_div_op", [(1, 0), (2, 0)])]
            if wrong:  # rows are summed before the exponential
                ops = [("tb_reduction_1_op", [(0, 0)]), ("tb_exp_op", [(0, 0)]), ("tb_div_op", [(2, 0), (1, 0)])]
            imap = (0, -1, -1)
            return ref[:2] + [first, {"op": "customized", "in": [[2, 0]],
                                      "plan": W._plan((m // mt, 1, 1), 1, [imap], (-1,), imap, ops)}]

    return ref, [candidate(rng.random() < 0.25) for _ in range(c["candidates"])]


# ---------------------------------------------------------------------------------------------
# state of a program
# ---------------------------------------------------------------------------------------------
_open = []  # graphs in the order they were built: the device arena they share is a stack


class _Graph:
    """A built graph.  It leaves the arena once nobody holds it any more -- neither the program's
    state nor a view of one of its tensors -- and everything built after it has left."""

    def __init__(self, spec):
        self.graph, self.tensors = G.build_from_spec(spec)
        self.entry = [self.graph, True]
        _open.append(self.entry)

    def __del__(self):
        self.entry[1] = False
        while _open and not _open[-1][1]:
            _open.pop()[0].close()


class _Memory:
    """A device tensor of the framework for torch.as_tensor: no copy."""

    def __init__(self, owner, tensor, fingerprint):
        self.owner = owner
        self.__cuda_array_interface__ = {
            "shape": tuple(tensor.dims), "typestr": "<i2" if fingerprint else "<f2",  # ring values are below 2^15
            "data": (tensor.device_ptr(fingerprint), False), "strides": None, "version": 2}


def _view(owner, tensor, fingerprint):
    return torch.as_tensor(_Memory(owner, tensor, fingerprint), device="cuda")


class _State:
    """What the program keeps between calls."""


# standard deviation of the values of input i
_STD = {"decode": [0.125] * 3, "split_kv": [0.125] * 3, "prefill": [0.125] * 3, "unfused_attention": [0.125] * 3,
        "matmul_op": [0.1, 0.1], "lora": [0.25, 0.02, 0.02, 0.02], "gated_mlp": [0.25, 0.02, 0.02, 0.02],
        "unfused_mlp": [0.25, 0.02, 0.02, 0.02]}


def _sinks(spec):
    """Operators whose results nobody in the graph consumes."""
    used = {ref[0] for op in spec for ref in op.get("in", [])}
    return [i for i in range(len(spec)) if i not in used]


def prepare(case, seed):
    G.set_smem_budget(1 << 20)
    s = _State()
    s.kind = case["kind"]
    s.seed = seed + 1
    if s.kind == "search":
        spec, s.candidate_specs = _search_specs(case, seed)
        s.reference = _Graph(spec)
        s.candidates = [_Graph(c) for c in s.candidate_specs] if case["built"] else None
        s.out = [_view(s.reference, s.reference.tensors[i][0], True) for i in _sinks(spec)]
    elif s.kind == "equivalence":
        s.mugraph, s.reference = (_Graph(spec) for spec in _specs(case))
        s.pair = s.mugraph.tensors[-1][0], s.reference.tensors[-1][0]
        s.out = [_view(s.mugraph, s.pair[0], True), _view(s.reference, s.pair[1], True)]
    else:
        spec, _ = _specs(case)
        s.program = _Graph(spec)
        gen = torch.Generator(device="cuda").manual_seed(seed)
        for i, std in enumerate(_STD[s.kind]):
            flat = _view(s.program, s.program.tensors[i][0], False).view(-1)
            for at in range(0, flat.numel(), 1 << 26):  # in pieces: the values are drawn in fp32
                part = flat[at:at + (1 << 26)]
                part.copy_(torch.randn(part.numel(), device="cuda", generator=gen).mul_(std))
        torch.cuda.synchronize()
        s.out = [_view(s.program, t, False) for i in _sinks(spec) for t in s.program.tensors[i]]
    return s


def run(s):
    if s.kind == "equivalence":
        s.mugraph.graph.fingerprint_seeded(s.seed)
        s.reference.graph.fingerprint_seeded(s.seed)
        return [s.pair[0].has_same_fingerprint(s.pair[1])] + s.out
    if s.kind == "search":
        if s.candidates is not None:
            graphs = [c.graph for c in s.candidates]
        else:
            graphs = [G.build_from_spec(spec)[0] for spec in s.candidate_specs]
        verdicts, _ = G.verify_batch_end(G.verify_batch_begin(graphs, s.reference.graph, s.seed))
        if s.candidates is None:
            for g in reversed(graphs):
                g.close()
        return [np.array(verdicts)] + s.out
    s.program.graph.execute_all()
    return s.out


# ---------------------------------------------------------------------------------------------
# work and tolerance
# ---------------------------------------------------------------------------------------------
def work(case):
    """Inputs read once, results written once; two operations per multiply-add of a matmul and one
    per element of the others."""
    c, k = case, case["kind"]
    if k in ("decode", "split_kv", "prefill", "unfused_attention", "equivalence"):
        if k == "prefill":
            b, m, s, hd = c["heads"], c["row_tile"] * c["row_blocks"], c["key_tile"] * c["loop"], c["head"]
        elif k == "unfused_attention":
            b, m, s, hd = c["heads"], c["rows"], c["keys"], c["head"]
        elif k == "equivalence":
            b, m, s, hd = c["heads"], c["rows"], c["key_tile"] * c["kv_blocks"] * c["loop"], c["head"]
        else:
            b, m, s, hd = c["groups"], c["rows"], c["key_tile"] * c["kv_blocks"] * c["loop"], 64
        out = b * m * hd * (c["kv_blocks"] if k == "decode" else 1)
        nbytes, flops = 2 * (b * m * hd + 2 * b * s * hd + out), b * m * s * (4 * hd + 3)
        return {"bytes": 2 * nbytes, "flops": 2 * flops} if k == "equivalence" else {"bytes": nbytes, "flops": flops}
    if k == "matmul_op":
        m, n, d = c["m"], c["col_tile"] * c["col_blocks"], c["k_tile"] * c["loop"]
        return {"bytes": 2 * (m * d + d * n + m * n), "flops": 2 * m * n * d}
    if k == "lora":
        m, n, d, r = c["m"], c["col_tile"] * c["col_blocks"], c["k_tile"] * c["loop"], c["rank"]
        return {"bytes": 2 * (m * d + d * n + d * r + r * n + m * n), "flops": 2 * m * (d * n + d * r + r * n)}
    if k in ("gated_mlp", "unfused_mlp"):
        m, d, h = (c["m"], c["d"], c["h"]) if k == "unfused_mlp" else (c["m"], 64 * c["d_blocks"], 64 * c["h_blocks"])
        return {"bytes": 2 * (2 * m * d + 3 * d * h), "flops": 6 * m * d * h + 2 * m * h}
    # search: the inputs are filled once (every candidate has the same), every candidate and the
    # reference graph multiply once and write their result
    m, d, h, n = (min(c["m"], 128) if c["family"] == "mlp" else c["m"]), c["k"], c["h"], c["n"]
    ins, macs, out = {
        "attention": (max(1, h // 64) * 64 * (m + 2 * n), max(1, h // 64) * m * n * 128, max(1, h // 64) * m * 64),
        "matmul_add": (m * d + d * n + m * n, m * n * d, m * n),
        "mlp": (m * d + d * h + h * n, m * h * (d + n), m * n),
        "row_softmax": (m * d + d * n, m * n * d, m * n)}[c["family"]]
    graphs = c["candidates"] + 1
    return {"bytes": 2 * (ins + graphs * out), "flops": 2 * macs * graphs}


def tolerance(case):
    if case["kind"] in ("search", "equivalence"):
        return "exact"  # whole numbers of a ring, and verdicts about them
    # fp16 results of fp32 sums, rounded to fp16 once per tile and per for-loop iteration: another
    # order of a sum moves a rounding by one unit in the last place (2^-11) here and there
    return {"rel": 2e-3}
