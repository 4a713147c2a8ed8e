"""The one-launch fingerprint matmul (operands reduced on the way into LDS), bit for bit."""
import numpy as np
import pytest

from helpers import FP_PQ, uniform_fp
from oracle import evaluate as orc
from test_gpu_fingerprint import _matmul_many

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shapes", [
    [(1, 1, 1, 1), (1, 17, 68, 4), (1, 64, 64, 64)],               # edges of a tile, one chunk of k
    [(2, 65, 60, 128), (1, 402, 64, 64)],                          # the last k of the 24-bit quotients
    [(1, 16, 64, 132), (3, 33, 132, 320)],                         # and the first beyond; two wavefronts share k
    [(1, 20, 72, 1024), (1, 64, 64, 1020)],                        # four of them
    [(2, 300, 700, 192), (1, 1030, 520, 60)],                      # a workgroup or more per compute unit
    [(1, 31, 33, 77), (2, 130, 65, 300), (1, 70, 1, 1023)],        # rows that are not whole 8-byte groups
], ids=lambda s: "+".join("x".join(map(str, t)) for t in s))
def test_direct_matmuls_match_oracle(rt, abi, shapes):
    ins, got = _matmul_many(abi, rt, shapes, lambda i, d: uniform_fp(d, 30 + i))
    for (A, B), C, s in zip(ins, got, shapes):
        np.testing.assert_array_equal(C, orc.fp_matmul(A, B), err_msg=str(s))


@pytest.mark.parametrize("k", [128, 1024])
def test_direct_matmul_of_every_ring_value_with_itself(rt, abi, k):
    """Sums of k equal products v * v for all v: the largest and smallest residues, squared."""
    per = 2048 // (k // 64)
    vals = np.arange(FP_PQ, dtype=np.int64)
    shapes = [(min(per, FP_PQ - at), 1, 4, k) for at in range(0, FP_PQ, per)]
    for lo in range(0, len(shapes), 40):
        part = shapes[lo:lo + 40]

        def fill(i, d):
            at = (lo + i % 100) * per
            return np.broadcast_to(vals[at:at + d[0], None, None], d).astype(np.uint16)

        _, got = _matmul_many(abi, rt, part, fill)
        for i, C in enumerate(got):
            v = vals[(lo + i) * per:][:C.shape[0], None, None]
            np.testing.assert_array_equal(C, np.broadcast_to(k * v * v % FP_PQ, C.shape))


@pytest.mark.parametrize("n", [4, 64, 6])  # whole groups of four, whole tiles, odd rows
def test_direct_matmul_of_every_16_bit_value(rt, abi, n):
    """Operands hold any 16-bit value, in the ring or past it, as in the other fingerprint kernels."""
    every = np.arange(65536, dtype=np.uint16)
    shapes = [(16, 64, n, 64), (18, 64, n, 60)]
    for flip in (False, True):  # every value as an element of A, and of B
        def fill(i, d, flip=flip):
            if (i >= 100) == flip:
                return np.resize(every, int(np.prod(d))).reshape(d)
            return uniform_fp(d, 3 + i)

        ins, got = _matmul_many(abi, rt, shapes, fill)
        for (A, B), C, s in zip(ins, got, shapes):
            np.testing.assert_array_equal(C, orc.fp_matmul(A % FP_PQ, B % FP_PQ), err_msg=str(s))


@pytest.mark.parametrize("b,m,n,k", [(1, 1, 1, 1025), (8, 96, 64, 1152), (1, 64, 64, 1088), (3, 7, 130, 2049), (1, 33, 5, 33000)])
def test_small_products_of_a_long_k(rt, abi, b, m, n, k):
    """Past the k of the one-launch kernel, as a graph's operator: on residue planes however small, for every
    16-bit value, and the same as the vector kernels."""
    from test_gpu_fingerprint import _graph_fp
    every = np.arange(65536, dtype=np.uint16)
    A, B = np.resize(every[::-1], b * m * k).reshape(b, m, k), uniform_fp((b, k, n), 8)
    spec = [{"op": "input", "dims": [b, m, k]}, {"op": "input", "dims": [b, k, n]}, {"op": "matmul", "in": [[0, 0], [1, 0]]}]
    got = _graph_fp(rt, spec, {0: A, 1: B})[2][0]
    np.testing.assert_array_equal(got, orc.fp_matmul(A % FP_PQ, B))
    assert abi.mi355_set_option(4, 1) == 0
    try:
        np.testing.assert_array_equal(got, _graph_fp(rt, spec, {0: A, 1: B})[2][0])
    finally:
        assert abi.mi355_set_option(4, 0) == 0
