"""Prepared operators (mi355_prepare / mi355_prepared_run, and KNCustomizedOp's kept launches): the launches
are recorded again when the options, the queue or the storage orders are no longer those they were recorded
under, and a plan that its fused kernel declines is recorded on the interpreter.  Pairs of operators
(mi355_prepare_two) with what they share besides: a queue's tickets, which a pair owns while it exists, and the
queue's memory for operand copies, where a gated MLP's product lies between its two launches."""
import ctypes

import numpy as np
import pytest

from attention_superoptimizer_amd import _native as N
from attention_superoptimizer_amd import graph as G
from attention_superoptimizer_amd import workloads as W
from helpers import assert_f16_close, normal_f16, uniform_fp
from oracle import evaluate as orc
from test_gpu_f16 import KERNEL_ATTENTION, KERNEL_COMBINE, KERNEL_GEMM, KERNEL_INTERP

pytestmark = pytest.mark.gpu
FORCE_INTERPRETER, GEMM_MODE = 1, 7


def _kernel():
    info = N.Mi355LaunchInfo()
    assert N.backend().mi355_last_launch(ctypes.byref(info)) == 0
    return info.kernel_id, info.workgroups


class Prepared:
    """The last operator of a spec, prepared through the C ABI."""

    def __init__(self, rt, abi, spec, fingerprint, seed=3, std=0.1):
        self.abi, self.fp = abi, fingerprint
        self.graph, self.vals = rt.build_from_spec(spec)
        self.ins = {}
        for i, op in enumerate(spec):
            if op["op"] == "input":
                self.ins[i] = uniform_fp(op["dims"], seed + i) if fingerprint else normal_f16(op["dims"], std, seed + i)
                t = self.vals[i][0]
                (t.write_fingerprint if fingerprint else t.write_data)(self.ins[i])
        self.want = orc.eval_graph(spec, "fp" if fingerprint else "f16", self.ins, threads=8)[-1]
        plan = self.graph.lowered(len(spec) - 1, fingerprint)
        ins = (ctypes.c_void_p * 4)(*[self.vals[a][b].device_ptr(fingerprint) for a, b in spec[-1]["in"]])
        outs = (ctypes.c_void_p * 4)(*[t.device_ptr(fingerprint) for t in self.vals[-1]])
        self.handle = ctypes.c_void_p()
        assert abi.mi355_prepare(ctypes.byref(plan), ins, outs, 1 if fingerprint else 0, ctypes.byref(self.handle)) == 0, N.last_error()

    def run(self):
        """One run; its outputs, checked against the oracle, and the kernel that made them."""
        for t in self.vals[-1]:
            if self.fp:
                t.write_fingerprint(np.full(t.dims, 7, np.uint16))
            else:
                t.write_data(np.full(t.dims, np.nan, np.float16))
        assert self.abi.mi355_prepared_run(self.handle) == 0, N.last_error()
        kernel = _kernel()
        assert self.abi.mi355_sync() == 0
        got = [t.read_fingerprint() if self.fp else t.read_data() for t in self.vals[-1]]
        for g, w in zip(got, self.want):
            if self.fp:
                np.testing.assert_array_equal(g, w)
            else:
                assert_f16_close(g, w, what=str(kernel))
        return kernel

    def close(self):
        assert self.abi.mi355_prepared_free(self.handle) == 0
        self.graph.close()


@pytest.fixture
def prepared(rt, abi):
    made = []

    def make(spec, fingerprint=False, **kw):
        made.append(Prepared(rt, abi, spec, fingerprint, **kw))
        return made[-1]

    yield make
    for p in reversed(made):
        p.close()
    for option in (FORCE_INTERPRETER, GEMM_MODE):
        assert abi.mi355_set_option(option, 0) == 0
    assert abi.mi355_queue_select(0) == 0


def test_options_set_later_hold(abi, prepared):
    p = prepared(W.config1_fused_matmul()[0], std=0.05)
    first = p.run()
    assert first[0] == KERNEL_GEMM and p.run() == first
    assert abi.mi355_set_option(GEMM_MODE, 1) == 0
    ranges = p.run()
    assert ranges[0] == KERNEL_GEMM and ranges != first
    assert abi.mi355_set_option(FORCE_INTERPRETER, 1) == 0
    assert p.run()[0] == KERNEL_INTERP
    assert abi.mi355_set_option(FORCE_INTERPRETER, 0) == 0 and abi.mi355_set_option(GEMM_MODE, 0) == 0
    assert p.run() == first


@pytest.mark.parametrize("fingerprint", [False, True], ids=["fp16", "fingerprint"])
def test_runs_from_several_queues(abi, prepared, fingerprint):
    """LoRA: two launches with the queue's scratch memory between them in fp16; both queues' runs are in
    flight together, from one record that changes hands."""
    spec = W.config4_lora()[0]
    a, b = prepared(spec, fingerprint, seed=3, std=0.05), prepared(spec, fingerprint, seed=50, std=0.05)
    for q in (0, 2, 1, 2, 0):
        assert abi.mi355_queue_select(q) == 0
        a.run()
    for _ in range(8):
        for p, q in ((a, 0), (b, 1)):
            assert abi.mi355_queue_select(q) == 0
            assert abi.mi355_prepared_run(p.handle) == 0
    assert abi.mi355_sync() == 0
    for p in (a, b):
        for t, w in zip(p.vals[-1], p.want):
            if fingerprint:
                np.testing.assert_array_equal(t.read_fingerprint(), w)
            else:
                assert_f16_close(t.read_data(), w)


def test_a_declined_plan_is_recorded_on_the_interpreter(abi, prepared):
    """Head size 128, 80-key tiles and the division: of the attention family, but no kernel of it holds the
    tile's operands."""
    ops = [("tb_matmul_op", [(0, 0), (1, 0)]), ("tb_exp_op", [(3, 0)]), ("tb_reduction_2_op", [(4, 0)]),
           ("tb_div_op", [(4, 0), (5, 0)]), ("tb_matmul_op", [(6, 0), (2, 0)])]
    plan = W._plan((2, 3, 1), 2, [(0, -1, -1), (0, 2, -1), (0, 1, -1)], (-1, 2, 1), (0, 2, -1), ops, dimx=128)
    spec = [W._inp([2, 16, 128]), W._inp([2, 128, 480], "DmemColumnMajor"), W._inp([2, 480, 128], "DmemColumnMajor"),
            {"op": "customized", "in": [[0, 0], [1, 0], [2, 0]], "plan": plan}]
    p = prepared(spec, std=0.1)
    first = p.run()
    assert first[0] == KERNEL_INTERP and p.run() == first
    whole = prepared(W.config2_gqa_decode()[0], std=0.125)  # (the same form on its kernel)
    assert whole.run()[0] == KERNEL_ATTENTION and p.run() == first


def test_a_changed_storage_order_is_recorded_again(rt):
    """The same operator object before and after a layout search turned its weights' storage order, with the
    launches kept from before."""
    spec, _ = W.tiled_matmul(16, 256, 512, (4, 1, 1), 4, (-1, -1, -1), (1, -1, -1), (1, -1, -1))
    ins = {0: normal_f16([16, 512], 0.1, 1), 1: normal_f16([512, 256], 0.1, 2)}
    want = orc.eval_graph(spec, "f16", ins, threads=8)[2][0]
    g, vals = rt.build_from_spec(spec)
    try:
        def check(order):
            assert vals[1][0].column_major == (order == 101)
            for i, a in ins.items():
                vals[i][0].write_data(a)
            for _ in range(2):
                vals[2][0].write_data(np.full(vals[2][0].dims, np.nan, np.float16))
                g.execute_all()
                assert_f16_close(vals[2][0].read_data(), want, what=f"weights in order {order}")

        check(101 if vals[1][0].column_major else 100)
        for order in (100, 101, 100):
            G.optimize_layout(g, lambda op, layouts: 1.0 if op == 2 and [x for x in layouts if x < 200] == [100, order, 100] else 2.0)
            check(order)
    finally:
        g.close()


# ---- pairs of operators ------------------------------------------------------------------------
class Pair:
    """The last two operators of a spec, prepared together; `want`: the bits the operators give one by one."""

    def __init__(self, rt, abi, spec, seed=3, std=0.125):
        self.abi, self.handle = abi, None
        self.graph, self.vals = rt.build_from_spec(spec)
        for i, op in enumerate(spec):
            if op["op"] == "input":
                self.vals[i][0].write_data(normal_f16(op["dims"], std if i == 0 else 0.05 if len(spec) == 6 else std, seed + i))
            else:
                self.graph.execute(i)
        self.made = self.vals[-2] + self.vals[-1]
        self.want = [t.read_data().view(np.uint16) for t in self.made]
        self.plans = [self.graph.lowered(i, False) for i in (len(spec) - 2, len(spec) - 1)]
        self.args = []
        for i in (-2, -1):
            self.args += [(ctypes.c_void_p * 4)(*[self.vals[a][b].device_ptr(False) for a, b in spec[i]["in"]]),
                          (ctypes.c_void_p * 4)(*[t.device_ptr(False) for t in self.vals[i]])]
        self.handle = self.prepare()

    def prepare(self):
        """One more handle."""
        handle = ctypes.c_void_p()
        assert self.abi.mi355_prepare_two(ctypes.byref(self.plans[0]), *self.args[:2], ctypes.byref(self.plans[1]), *self.args[2:], 0,
                                          ctypes.byref(handle)) == 0, N.last_error()
        return handle

    def clear(self):
        for t in self.made:
            t.write_data(np.full(t.dims, -7, np.float16))

    def enqueue(self, handle=None):
        assert self.abi.mi355_prepared_run(handle or self.handle) == 0, N.last_error()
        return _kernel()[0]

    def check(self, what=""):
        assert self.abi.mi355_sync() == 0
        for t, w in zip(self.made, self.want):
            np.testing.assert_array_equal(t.read_data().view(np.uint16), w, err_msg=what)

    def run(self, handle=None):
        self.clear()
        kernel = self.enqueue(handle)
        self.check(str(kernel))
        return kernel

    def free(self, handle=None):
        if handle is not None or self.handle is not None:
            assert self.abi.mi355_prepared_free(handle or self.handle) == 0
        if handle is None:
            self.handle = None

    def close(self):
        self.free()
        self.graph.close()


@pytest.fixture
def pairs(rt, abi):
    made = []

    def make(spec, **kw):
        made.append(Pair(rt, abi, spec, **kw))
        return made[-1]

    yield make
    assert abi.mi355_queue_select(0) == 0
    for p in reversed(made):
        p.close()
    for option in (FORCE_INTERPRETER, GEMM_MODE):
        assert abi.mi355_set_option(option, 0) == 0


def _split_kv(groups=3, rows=16, blocks=4):
    """Pieces of several workgroups: the last of a row block's folds them."""
    return W.gqa_inc_decode(groups=groups, rows=rows, seq=64 * blocks * 3, kv_blocks=blocks, F=3)[0]


def _gated(h=1792):
    return W.config5_gated_mlp(m=8, d=256, h=h, grid1=h // 64, F1=4, grid2=4, F2=h // 64)[0]


def test_options_set_later_hold_for_pairs(abi, pairs):
    p = pairs(_split_kv())
    assert p.run() == KERNEL_ATTENTION
    for _ in range(2):
        assert abi.mi355_set_option(FORCE_INTERPRETER, 1) == 0
        p.clear()
        assert p.enqueue() == KERNEL_INTERP and abi.mi355_sync() == 0
        for t, w in zip(p.made, p.want):
            assert_f16_close(t.read_data(), w.view(np.float16))
        assert abi.mi355_set_option(FORCE_INTERPRETER, 0) == 0
        for _ in range(3):
            assert p.run() == KERNEL_ATTENTION
    g = pairs(_gated())
    for mode in (0, 1, 2, 0):  # (the kernel of both products)
        assert abi.mi355_set_option(GEMM_MODE, mode) == 0
        assert g.run() == KERNEL_GEMM and p.run() == KERNEL_ATTENTION


@pytest.mark.parametrize("spec", [_split_kv, _gated])
def test_pairs_run_from_several_queues(abi, pairs, spec):
    """One handle that changes hands between queues, and handles of two queues in flight together."""
    a, b = pairs(spec(), seed=3), pairs(spec(), seed=50)
    for q in (0, 2, 1, 2, 0):
        assert abi.mi355_queue_select(q) == 0
        a.run()
    for x in (a, b):
        x.clear()
    for _ in range(8):
        for p, q in ((a, 0), (b, 1)):
            assert abi.mi355_queue_select(q) == 0
            p.enqueue()
    a.check(), b.check()
    for x in (a, b):
        x.clear()
    for _ in range(8):  # ... and one behind the other in one queue
        for p in (a, b):
            p.enqueue()
    a.check(), b.check()


def test_tickets_go_to_the_next_pair(pairs):
    """A pair takes the tickets that another gave back with launches of it still in the queue."""
    a, b = pairs(_split_kv(), seed=3), pairs(_split_kv(groups=5, blocks=6), seed=50)
    b.free()
    for _ in range(4):
        a.clear(), b.clear()
        for _ in range(16):
            assert a.enqueue() == KERNEL_ATTENTION
        a.free()
        b.handle = b.prepare()
        for _ in range(16):
            assert b.enqueue() == KERNEL_ATTENTION
        b.free()
        a.handle = a.prepare()
        assert a.enqueue() == KERNEL_ATTENTION
        a.check(), b.check()


def test_without_tickets_left_there_are_two_launches(pairs):
    """65,536 ints in units of 64 for each queue: 1024 pairs at most have some."""
    p = pairs(_split_kv())
    p.free()
    handles = []
    try:
        while len(handles) < 1025 and (not handles or p.enqueue(handles[-1]) == KERNEL_ATTENTION):
            handles.append(p.prepare())
        assert 512 < len(handles) and p.run(handles[-1]) == KERNEL_COMBINE and p.run(handles[0]) == KERNEL_ATTENTION
        p.free(handles.pop(7))
        handles.append(p.prepare())  # (in the place that is free again)
        assert p.run(handles[-1]) == KERNEL_ATTENTION and p.run(handles[-2]) == KERNEL_COMBINE
    finally:
        for h in handles:
            p.free(h)


def test_gated_pairs_beside_operand_copies(rt, abi, pairs):
    """A matmul that copies its operand writes the queue's memory that a gated pair's product passes through."""
    a, b = pairs(_gated(), seed=3), pairs(_gated(h=2048), seed=50)
    m, n, k = 563, 6177, 3520
    g = G.KNGraph()
    try:
        A, B = g.new_input((1, m, k), layout="DmemColumnMajor"), g.new_input((1, k, n), layout="DmemRowMajor")
        C = g.matmul(A, B)
        A.write_data(normal_f16([1, m, k], 0.1, 1)), B.write_data(normal_f16([1, k, n], 0.1, 2))
        g.execute(2)
        want = C.read_data().view(np.uint16)
        a.clear(), b.clear()
        C.write_data(np.full(C.dims, -7, np.float16))
        for _ in range(3):
            for p in (a, b):
                p.enqueue()
                g.execute(2)
        a.check(), b.check()
        np.testing.assert_array_equal(C.read_data().view(np.uint16), want)
    finally:
        g.close()


def test_a_changed_storage_order_is_recorded_again_for_pairs(rt):
    """The pair that execute_all keeps, before and after a layout search turned the keys' and values' storage order."""
    spec = _split_kv()
    ins = [normal_f16(op["dims"], 0.125, 3 + i) for i, op in enumerate(spec[:3])]
    want = orc.eval_graph(spec, "f16", dict(enumerate(ins)), threads=8)[-1][0]
    g, vals = rt.build_from_spec(spec)
    try:
        def check(order):
            assert [vals[i][0].column_major for i in (1, 2)] == [order == 101] * 2
            for i, a in enumerate(ins):
                vals[i][0].write_data(a)
            for _ in range(3):
                for t in vals[3] + vals[4]:
                    t.write_data(np.full(t.dims, np.nan, np.float16))
                g.execute_all()
                assert _kernel()[0] == KERNEL_ATTENTION
                assert_f16_close(vals[4][0].read_data(), want, what=f"keys and values in order {order}")

        check(101 if vals[1][0].column_major else 100)
        for order in (100, 101, 100):
            wanted = {3: [100, order, order, 100, 100], 4: [100, 100, 100]}
            G.optimize_layout(g, lambda op, layouts: 1.0 if wanted.get(op) == [x for x in layouts if x < 200] else 2.0)
            check(order)
    finally:
        g.close()
