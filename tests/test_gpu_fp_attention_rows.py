"""The fingerprints of the un-fused attention graph in one launch: every one of its tensors, bit for bit what the
operators leave one by one."""
import ctypes

import numpy as np
import pytest

from helpers import uniform_fp

pytestmark = pytest.mark.gpu


def _spec(b, m, n, d, dv):
    from attention_superoptimizer_amd import workloads as W
    return W.attention_reference([b, m, d], [b, d, n], [b, n, dv])


@pytest.mark.parametrize("b,m,n,d,dv,taken", [
    (1, 1, 8, 4, 4, 1), (1, 16, 64, 64, 64, 1), (2, 17, 72, 64, 60, 1),     # edges of a chunk, of a row group
    (1, 65, 1000, 60, 20, 1), (3, 33, 136, 32, 16, 1), (2, 16, 264, 64, 64, 1),  # eight and four wavefronts to 16 rows
    (130, 64, 64, 64, 64, 1), (40, 200, 200, 64, 64, 1), (257, 7, 1000, 8, 64, 1),  # eight to 32 rows
    (1, 16, 20, 64, 64, 0), (1, 16, 64, 68, 64, 0), (1, 16, 64, 64, 66, 0), (1, 16, 2048, 64, 64, 0)])  # left to the operators
def test_every_tensor_matches_the_operators(rt, abi, b, m, n, d, dv, taken):
    spec = _spec(b, m, n, d, dv)
    ins = [uniform_fp(spec[i]["dims"], 7 + i) for i in range(3)]
    # (any 16-bit value is an operand: every one of them in V, the largest in K)
    ins[2] = np.resize(np.arange(65536, dtype=np.uint16)[::-3], spec[2]["dims"])
    ins[1].flat[::7] = 65535
    one, ops = rt.build_from_spec(spec), rt.build_from_spec(spec)
    try:
        for vals in (one[1], ops[1]):
            for i, x in enumerate(ins):
                vals[i][0].write_fingerprint(x)
        for i in range(3, len(spec)):
            one[1][i][0].write_fingerprint(np.full_like(one[1][i][0].read_fingerprint(), 12345))
            ops[0].fingerprint(i)
        got = ctypes.c_int(7)
        assert abi.mi355_fp_attention_rows(*[one[1][i][0].device_ptr(True) for i in range(8)], b, m, n, d, dv,
                                           ctypes.byref(got)) == 0
        assert got.value == taken
        for i in range(3, len(spec)):
            want = ops[1][i][0].read_fingerprint() if taken else 12345
            np.testing.assert_array_equal(one[1][i][0].read_fingerprint(), want, err_msg=spec[i]["op"])
    finally:
        ops[0].close()  # (the arena is a stack)
        one[0].close()


@pytest.mark.parametrize("b,m,n,d,dv", [(4, 48, 320, 64, 64), (2, 16, 12, 64, 64)])
def test_a_graph_takes_it(rt, b, m, n, d, dv):
    """fingerprint_seeded of the graph, in one launch and not, against its operators."""
    spec = _spec(b, m, n, d, dv)
    one, ops = rt.build_from_spec(spec), rt.build_from_spec(spec)
    try:
        one[0].fingerprint_seeded(3)
        for i in range(3):
            ops[1][i][0].write_fingerprint(one[1][i][0].read_fingerprint())
        for i in range(3, len(spec)):
            ops[0].fingerprint(i)
            np.testing.assert_array_equal(one[1][i][0].read_fingerprint(), ops[1][i][0].read_fingerprint())
    finally:
        ops[0].close()  # (the arena is a stack)
        one[0].close()


def test_no_place_for_the_answer(rt, abi):
    assert abi.mi355_fp_attention_rows(*[None] * 8, 1, 16, 64, 64, 64, None) != 0
