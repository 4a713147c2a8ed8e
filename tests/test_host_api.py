"""Host-side logic of the product without a GPU: graph construction through the
mirage:: API (host-only runtime), lowering against the oracle's restatement, the
soft-failure contract, the LIFO arena, and the C ABI's symbols."""
import ctypes
import gc
import os
import re
import subprocess
import sys
import weakref

import numpy as np
import pytest

from helpers import load_gqa_fixture
from oracle import lowering
from attention_superoptimizer_amd import _native as N
from attention_superoptimizer_amd import graph as G
from attention_superoptimizer_amd import workloads as W

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(autouse=True)
def _budget():
    G.set_smem_budget(1 << 20)
    yield
    G.set_smem_budget(96 * 1024)


def _compare_lowering(spec):
    g, vals = G.build_from_spec(spec)
    try:
        for i, op in enumerate(spec):
            if op["op"] != "customized":
                continue
            p = g.lowered(i, True)
            ins = [vals[a][b] for a, b in op["in"]]
            tg = lowering.build_tb_graph(op["plan"], [list(t.dims) for t in ins],
                                         [t.layout for t in ins], 1 << 20)
            types, params = lowering.lower(tg)
            assert list(p.operator_types[:p.num_operators]) == types
            assert list(p.parameters[:p.num_parameters]) == params
            assert p.smem_bytes == tg.smem_offset
            assert [list(t.dims) for t in vals[i]] == lowering.output_dims(tg)
            assert list(p.grid_dim) == op["plan"]["grid_dim"]
            assert p.forloop_range == op["plan"]["forloop_range"]
    finally:
        g.close()


@pytest.mark.parametrize("name", sorted(W.REFERENCE_EXAMPLES))
def test_lowering_matches_oracle_examples(name):
    _compare_lowering(W.REFERENCE_EXAMPLES[name][0])


@pytest.mark.parametrize("name", sorted(W.BASELINE_CONFIGS))
def test_lowering_matches_oracle_configs(name):
    _compare_lowering(W.BASELINE_CONFIGS[name]()[0])


def test_lowering_matches_fixture_graphs():
    fx = load_gqa_fixture()
    for spec in fx["generated_graphs"]:
        g, vals = G.build_from_spec(spec)
        try:
            for i, op in enumerate(spec):
                assert [list(t.dims) for t in vals[i]] == op["out_dims"]
                if op["op"] == "customized":   # the reference recorded its own smem_offset
                    assert g.lowered(i, True).smem_bytes == op["smem_offset"]
        finally:
            g.close()
    _compare_lowering(fx["generated_graphs"][0])


def test_program_sizes_quoted_for_the_reference_plans():
    """GQA single-op plan = 3*19+6+2+5+9+6+17 = 102 ints; LoRA = 4*19+6+7+7+6+17 = 119"""
    g, _ = G.build_from_spec(W.config2_gqa_decode()[0])
    assert g.lowered(3).num_parameters == 102
    g.close()
    g, _ = G.build_from_spec(W.REFERENCE_EXAMPLES["lora"][0])
    assert g.lowered(4).num_parameters == 119
    g.close()


def test_shape_inference_and_soft_failures():
    g = G.KNGraph()
    try:
        A = g.new_input((2, 8, 16))
        B = g.new_input((2, 16, 4))
        C = g.matmul(A, B)
        assert C.dims == (2, 8, 4) and C.layout == 100          # outputs are row-major
        assert g.reduction(C, 2).dims == (2, 8, 1)
        assert g.reduction(C, 1, 4).dims == (2, 4, 4)
        S = g.new_input((2, 8, 1))
        assert g.div(C, S).dims == (2, 8, 4)
        n = g.num_operators
        with pytest.raises(G.InfeasibleOperator):
            g.matmul(A, C)                                       # inner dims differ
        with pytest.raises(G.InfeasibleOperator):
            g.matmul(A, g.new_input((3, 16, 4)))                 # batch dims differ
        with pytest.raises(G.InfeasibleOperator):
            g.add(C, g.new_input((2, 8, 3)))                     # not broadcastable
        with pytest.raises(G.InfeasibleOperator):
            g.reduction(C, 3)                                    # dim out of range
        with pytest.raises(G.InfeasibleOperator):
            g.reduction(C, 2, 3)                                 # 4 % 3 != 0
        assert g.num_operators == n + 2                          # only the two inputs were added
    finally:
        g.close()


def test_arena_is_lifo_and_bounded():
    rt = N.runtime()
    base = rt.mirage_arena_offset()
    g = G.KNGraph()
    A = g.new_input((4, 100, 33))
    nbytes = (4 * 100 * 33 * 2 + 15) // 16 * 16
    assert rt.mirage_arena_offset() == base + 2 * nbytes         # data + fingerprint buffers
    assert A.device_ptr(True) - A.device_ptr(False) == nbytes
    g.exp(A)
    assert rt.mirage_arena_offset() == base + 4 * nbytes
    g.pop_operator()
    assert rt.mirage_arena_offset() == base + 2 * nbytes
    with pytest.raises(G.InfeasibleOperator):                    # larger than the whole arena
        g.new_input((1 << 15, 1 << 15, 1 << 5))
    g.close()
    assert rt.mirage_arena_offset() == base


def test_smem_budget_is_enforced_by_default():
    """the reference's 96 KB cap: config C2 does not fit it, the spec-decode example does"""
    G.set_smem_budget(96 * 1024)
    g, _ = G.build_from_spec(W.REFERENCE_EXAMPLES["group_query_attn_spec_decode"][0])
    g.close()
    code = ("import os; os.environ['MIRAGE_HOST_ONLY']='1'\n"
            "from attention_superoptimizer_amd import graph as G, workloads as W\n"
            "G.build_from_spec(W.config2_gqa_decode()[0])\n")
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True)
    assert r.returncode != 0 and "infeasible" in r.stderr


def test_device_work_fails_loudly_without_a_gpu():
    if os.path.exists("/dev/kfd"):
        pytest.skip("a GPU is present")
    code = ("import os; os.environ['MIRAGE_HOST_ONLY']='1'\n"
            "from attention_superoptimizer_amd import graph as G\n"
            "g=G.KNGraph(); A=g.new_input((4,4)); g.fingerprint(0)\n")
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True)
    assert r.returncode != 0 and "host-only" in r.stderr
    # the two-call verification hands work to threads: it must refuse before starting any
    code = ("import os; os.environ['MIRAGE_HOST_ONLY']='1'\n"
            "from attention_superoptimizer_amd import graph as G\n"
            "g=G.KNGraph(); A=g.new_input((4,4)); r=G.KNGraph(); r.new_input((4,4))\n"
            "G.verify_batch_begin([g], r, 1)\n")
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True)
    assert r.returncode != 0 and "host-only" in r.stderr
    code = ("import os; os.environ.pop('MIRAGE_HOST_ONLY', None)\n"
            "from attention_superoptimizer_amd import graph as G\n"
            "g=G.KNGraph(); g.new_input((4,4))\n")
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True,
                       env={k: v for k, v in os.environ.items() if k != "MIRAGE_HOST_ONLY"})
    assert r.returncode != 0 and "cannot initialise the MI355X backend" in r.stderr


def test_abi_exports_every_declared_symbol():
    header = open(os.path.join(ROOT, "include", "mi355_abi.h")).read()
    declared = set(re.findall(r"\b(mi355_[a-z0-9_]+)\s*\(", header))
    assert declared, "no declarations found"
    lib = N.backend()
    for name in sorted(declared):
        assert hasattr(lib, name), f"{name} is declared but not exported"
    assert declared == set(N.ABI), (declared ^ set(N.ABI))
    # no compute without a device: entry points refuse instead of crashing
    if not os.path.exists("/dev/kfd"):
        assert lib.mi355_is_initialised() == 0
        assert lib.mi355_sync() == -5
        assert b"mi355_init" in lib.mi355_last_error()


def test_plan_extents_and_validation():
    ab = N.backend()
    g, vals = G.build_from_spec(W.config1_fused_matmul()[0])
    p = g.lowered(2, True)
    ie, oe = (ctypes.c_longlong * 4)(), (ctypes.c_longlong * 4)()
    l1, l2 = ctypes.c_int(), ctypes.c_int()
    assert ab.mi355_plan_extents(ctypes.byref(p), ie, oe, ctypes.byref(l1), ctypes.byref(l2)) == 0
    assert list(ie[:2]) == [64 * 1024, 1024 * 1024] and oe[0] == 64 * 1024
    assert 0 < l1.value <= 160 * 1024 and 0 < l2.value <= 160 * 1024
    p.parameters[13] = 512                       # claim the A matrix has 512 columns
    assert ab.mi355_plan_extents(ctypes.byref(p), ie, oe, None, None) == -3
    assert b"walks outside" in ab.mi355_last_error()
    p = g.lowered(2, True)
    p.num_parameters -= 1
    assert ab.mi355_plan_extents(ctypes.byref(p), ie, oe, None, None) == -3
    p = g.lowered(2, True)
    p.operator_types[2] = 2050
    assert ab.mi355_plan_extents(ctypes.byref(p), ie, oe, None, None) == -4
    g.close()


def test_verify_ring_never_hands_out_what_a_live_batch_owns():
    """Compare-slot ranges and mark pairs of verification batches in flight (verify.cc): a new
    batch never overlaps a live one; ranges and marks come back when a batch ends; the 33rd
    batch in flight, or a range no free stretch can hold, is refused."""
    import ctypes
    from attention_superoptimizer_amd import _native as N
    rt = N.runtime()
    ring = ctypes.c_void_p(rt.mirage_verify_ring_create())
    try:
        first, ticket = ctypes.c_int(), ctypes.c_int()
        live = {}

        def acquire(n):
            rc = rt.mirage_verify_ring_acquire(ring, n, ctypes.byref(first), ctypes.byref(ticket))
            if rc != 0:
                return None
            for f, c in live.values():
                assert n == 0 or c == 0 or first.value >= f + c or f >= first.value + n, "overlap"
            assert ticket.value not in live and 0 <= ticket.value < 32
            assert 0 <= first.value and first.value + n <= 65536
            live[ticket.value] = (first.value, n)
            return ticket.value

        def release(t):
            rt.mirage_verify_ring_release(ring, t)
            del live[t]

        # three batches of 30,000 slots: the third does not fit until the first has ended
        a, b = acquire(30000), acquire(30000)
        assert a is not None and b is not None
        assert acquire(30000) is None
        release(a)
        c = acquire(30000)
        assert c is not None and live[c][0] == 0          # wrapped into the freed stretch, not onto b
        assert acquire(10000) is None                     # 5,536 free slots at the end only
        d = acquire(5000)
        assert d is not None and live[d][0] == 60000
        for t in list(live):
            release(t)
        # 32 batches in flight use every mark pair; the 33rd is refused until one ends
        ts = [acquire(16) for _ in range(32)]
        assert None not in ts and len(set(ts)) == 32
        assert acquire(16) is None
        release(ts[7])
        assert acquire(16) == ts[7]
        # long run of begin / end with a few in flight: wraps the ring many times
        for t in list(live):
            release(t)
        import random
        rnd = random.Random(5)
        order = []
        for _ in range(2000):
            if len(order) < 4 or (len(order) < 20 and rnd.random() < 0.5):
                t = acquire(rnd.choice([0, 1, 64, 4096, 9000]))
                if t is not None:
                    order.append(t)
                    continue
            release(order.pop(0))
        assert acquire(65537) is None
    finally:
        rt.mirage_verify_ring_destroy(ring)


# ---- the two readers of a graph spec: the extension, and the ctypes calls it stands in for ----------
def _readers():
    if N.spec() is None:
        pytest.skip("built without the extension")
    return [lambda g, s: N.spec().build(g._g.value, s, G.DTensor, G.DMEM_LAYOUT, G.SMEM_LAYOUT, G.KN_OP, G.TB_OP,
                                        G.InfeasibleOperator), G._build_in_python]


def _outcome(read, spec):
    """The graph a reader builds, as JSON and tensors without their ids, or the error it raises."""
    g = G.KNGraph()
    try:
        vals = read(g, spec)
        text = re.sub(r'"guid":-?\d+', '"guid":0', g.to_json())
        return text, [[(t.dims, t.data_type, t.layout) for t in v] for v in vals]
    except Exception as e:  # noqa: BLE001 -- the kind of error is the outcome
        return type(e)
    finally:
        g.close()


def _all_specs():
    for name in sorted(W.REFERENCE_EXAMPLES):
        yield from W.REFERENCE_EXAMPLES[name]
    for name in sorted(W.BASELINE_CONFIGS):
        yield from (s for s in W.BASELINE_CONFIGS[name]() if s is not None)
    yield from load_gqa_fixture()["generated_graphs"]


def test_negative_counts_are_none():
    """A plan whose counts are negative has no operators (no inputs): it builds an operator without results, in a
    process that goes on."""
    code = """
import ctypes
from attention_superoptimizer_amd import graph as G, _native as N, workloads as W
spec, _ = W.tiled_matmul(128, 256, 256, (2, 4, 1), 4, (0, -1, -1), (-1, 1, -1), (0, 1, -1))
with G.KNGraph() as g:
    ins = (ctypes.c_void_p * 2)(g.new_input((128, 256))._h, g.new_input((256, 256))._h)
    outs = (ctypes.c_void_p * 4)()
    for inputs in (2, 0, -1):
        cp = G._c_plan(spec[2]["plan"])
        cp.num_ops, cp.num_inputs = -1, inputs
        print(N.runtime().mirage_graph_customized(g._g, ins, inputs, ctypes.byref(cp), outs, 4), end=" ")
"""
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, env=dict(os.environ, MIRAGE_HOST_ONLY="1"))
    assert r.returncode == 0 and r.stdout.split() == ["0", "0", "0"], r.stderr


def test_extension_makes_whole_tensors():
    """Tensors made without their __init__ are like any others; a derived class has its own called."""
    native, _ = _readers()
    made = []

    class Counted(G.DTensor):
        def __init__(self, *args):
            made.append(args)
            super().__init__(*args)

    spec = next(_all_specs())
    with G.KNGraph() as g:
        first = native(g, spec)[0][0]
        assert (first.dims, first.data_type, first.guid, first.layout) == first._info()
        gone, refs = weakref.ref(first), sys.getrefcount(G.DTensor)
        assert gc.is_tracked(first)
        del first
        gc.collect()
        assert gone() is None and sys.getrefcount(G.DTensor) <= refs
    with G.KNGraph() as g:
        vals = N.spec().build(g._g.value, spec, Counted, G.DMEM_LAYOUT, G.SMEM_LAYOUT, G.KN_OP, G.TB_OP, G.InfeasibleOperator)
        assert len(made) == sum(len(v) for v in vals) and all(type(t) is Counted for v in vals for t in v)


def _build_as(cls):
    spec = next(_all_specs())
    with G.KNGraph() as g:
        vals = N.spec().build(g._g.value, spec, cls, G.DMEM_LAYOUT, G.SMEM_LAYOUT, G.KN_OP, G.TB_OP, G.InfeasibleOperator)
        return [(type(t), {n for n in ("_h", "dims", "data_type", "guid", "more") if hasattr(t, n)}) for v in vals for t in v]


def test_extension_calls_an_init_that_does_more(monkeypatch):
    """Only the __init__ that the class says keeps its arguments is passed by."""
    _readers()
    made = []

    def slots(*more):
        def init(self, handle, dims, data_type, guid):
            made.append(guid)
            self._h, self.dims, self.data_type, self.guid = handle, dims, data_type, guid
            for name in more:
                setattr(self, name, 0)
        return {"__slots__": ("_h", "dims", "data_type", "guid", *more), "__init__": init}

    kept = {"_h", "dims", "data_type", "guid"}
    assert all(t == (G.DTensor, kept) for t in _build_as(G.DTensor)) and not made
    other, wider = type("Other", (), slots()), type("Wider", (), slots("more"))
    promising = slots("more")
    promising = type("Promising", (), dict(promising, _keeping_init=promising["__init__"]))
    for cls, names in ((other, kept), (wider, kept | {"more"}), (promising, kept | {"more"})):
        made.clear()
        tensors = _build_as(cls)
        assert len(made) == len(tensors) and all(t == (cls, names) for t in tensors)
    made.clear()
    keep = G.DTensor.__init__
    monkeypatch.setattr(G.DTensor, "__init__", lambda self, *args: (made.append(args), keep(self, *args))[1])
    tensors = _build_as(G.DTensor)
    assert len(made) == len(tensors) and all(t == (G.DTensor, kept) for t in tensors)


def test_readers_build_the_same_graphs():
    native, python = _readers()
    n = 0
    for spec in _all_specs():
        want = _outcome(python, spec)
        assert not isinstance(want, type), want
        assert _outcome(native, spec) == want
        n += 1
    assert n > 60


@pytest.mark.parametrize("change", [
    {}, {"block_dim": [64, 2, 1]}, {"reduction_dimx": 16}, {"input_smem_layouts": []}, {"input_smem_layouts": None},
    {"input_smem_layouts": ["SmemColumnMajor", "SmemRowMajor"]}, {"input_smem_layouts": [201, 299]},
    {"grid_dim": (4, 1, 1)}, {"input_map": ((-1, -1, -1), (1, -1, -1))},      # tuples as well as lists
    {"grid_dim": [4, 1]}, {"input_map": [[-1, -1], [1, -1, -1]]}, {"input_map": [[-1, -1, -1]] * 5}, {"forloop_dim": [1]},
    {"forloop_range": None}, {"forloop_range": "4"}, {"forloop_range": 8}, {"ops": [["tb_nothing_op", [[0, 0]]]]},
    {"ops": [["tb_matmul_op", [[0, 0], [1, 0], [0, 0]]]]}, {"ops": [["tb_exp_op", [[0, 0]]]] * 17}, {"ops": [[2003, [[0, 0], [1, 0]]]]},
    {"ops": [["tb_matmul_op"]]}, {"ops": [["tb_matmul_op", [[0, 0], [1, 0]], 0]]}, {"ops": [["tb_matmul_op", [[0, 0, 0], [1, 0]]]]},
    {"ops": [["tb_matmul_op", [[0], [1, 0]]]]}, {"ops": [[]]}, {"input_smem_layouts": ["SmemNothing", "SmemRowMajor"]}, {"output_map": 1},
])
def test_readers_take_the_same_plans(change):
    native, python = _readers()
    spec, _ = W.tiled_matmul(16, 256, 256, (4, 1, 1), 4, (-1, -1, -1), (1, -1, -1), (1, -1, -1))
    spec = [dict(op) for op in spec]
    spec[2]["plan"] = {**spec[2]["plan"], **change}
    assert _outcome(native, spec) == _outcome(python, spec)


@pytest.mark.parametrize("key", ["grid_dim", "output_map", "forloop_range", "input_map", "forloop_dim", "ops"])
def test_readers_miss_the_same_keys(key):
    native, python = _readers()
    spec, _ = W.tiled_matmul(16, 256, 256, (4, 1, 1), 4, (-1, -1, -1), (1, -1, -1), (1, -1, -1))
    spec = [dict(op) for op in spec]
    spec[2]["plan"] = {k: v for k, v in spec[2]["plan"].items() if k != key}
    assert _outcome(native, spec) == _outcome(python, spec) == KeyError


@pytest.mark.parametrize("op", [
    {"op": "exp", "in": [[0, 0]]}, {"op": "exp", "in": [[-1, -1]]}, {"op": "mul", "in": [[0, 0], [0, 0]]},
    {"op": "reduction", "in": [[0, 0]], "dim": 1}, {"op": "reduction", "in": [[0, 0]], "dim": 1, "size": 64},
    {"op": "reduction", "in": [[0, 0]]}, {"op": "exp", "in": [[1, 0]]}, {"op": "exp", "in": [[0, 1]]}, {"op": "exp"},
    {"op": "matmul", "in": [[0, 0]]}, {"op": "matmul", "in": [[0, 0], [0, 0]]}, {"op": "nothing", "in": [[0, 0]]},
    {"op": "input", "dims": [4, 4], "layout": "DmemNothing"}, {"op": "input", "dims": [2.5]}, {},
])
def test_readers_take_the_same_operators(op):
    native, python = _readers()
    spec = [{"op": "input", "dims": [64, 256]}, op]
    assert _outcome(native, spec) == _outcome(python, spec)


def test_a_package_without_the_extension_builds_graphs(monkeypatch):
    """`_spec` is built only where Python's headers are (and by CMake only then): the package runs without."""
    spec = W.config2_gqa_decode()[0]
    want = _outcome(lambda g, s: G.build_from_spec(s, g)[1], spec)
    import importlib

    def absent(name, *a):
        raise ModuleNotFoundError(f"No module named {name!r}", name=name)

    monkeypatch.setattr(N, "_spec", None)
    monkeypatch.setattr(importlib, "import_module", absent)
    assert N.spec() is None
    assert _outcome(lambda g, s: G.build_from_spec(s, g)[1], spec) == want
    assert N.spec() is None
    monkeypatch.setattr(N, "_spec", None)

    def broken(name, *a):
        raise ImportError(f"{name}: undefined symbol")

    monkeypatch.setattr(importlib, "import_module", broken)
    with pytest.raises(ImportError):  # one that is there but does not load is not passed over
        N.spec()
