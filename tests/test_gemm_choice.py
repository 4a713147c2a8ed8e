"""The kernel a kernel-level fp16 matmul is given (csrc/backend/f16_gemm_choice.h), without a device."""
import os
import random
import subprocess

import pytest

from test_gpu_matmul_two import COL, SHAPES, TAKEN

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
STAGED, DIRECT, WAVES = 0, 1, 2
SCRATCH, COPIES = 64 << 20, 128 << 20  # what a queue has


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    exe = tmp_path_factory.mktemp("choice") / "gemm_choice"
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-I",
                           os.path.join(ROOT, "attention_superoptimizer_amd", "csrc", "backend"), "-o", str(exe),
                           os.path.join(ROOT, "tests", "cpp", "gemm_choice.cc")])
    return exe


@pytest.fixture(scope="module")
def choose(exe):
    def one(batch, m, n, k, a_cm=0, b_cm=1, aligned=1, scratch=SCRATCH, copies=COPIES):
        out = subprocess.run([str(exe)], input=f"{batch} {m} {n} {k} {a_cm} {b_cm} {aligned} {scratch} {copies}\n", capture_output=True,
                             text=True, check=True).stdout.split()
        return dict(zip(("route", "copy_a", "copy_b", "kind", "bm", "bn", "ksplit"), [out[0]] + [int(x) for x in out[1:7]]))

    return one


# microseconds measured on the 256 x 256 kernel and on the best-expected tiles
@pytest.mark.parametrize("shape,b_cm,big,tiles", [
    ((32, 2048, 2048, 128), 1, 103, 113),   # the scores of a prefill at head size 128
    ((32, 2048, 2048, 32), 1, 67, 82),
    ((32, 2048, 2048, 384), 1, 173, 203),
    ((1, 4096, 4096, 32), 1, 10, 12),
    ((1, 4096, 4096, 1024), 1, 38, 49),
    ((8, 2048, 2048, 512), 1, 47, 57),
    ((32, 500, 1000, 1024), 1, 40, 50),
    ((12, 1040, 1040, 128), 1, 21, 14),     # two rounds of 256 tiles, the second almost empty
    ((12, 1040, 1040, 1024), 1, 62, 44),
    ((4, 1024, 1024, 1024), 1, 27, 13),     # far fewer tiles than compute units
    ((200, 130, 130, 64), 1, 10, 8),        # tiles mostly padding
    ((8, 2048, 2048, 128), 0, 33, 27),      # B would have to be copied
    ((32, 500, 1000, 1024), 0, 79, 54),
    ((1, 4096, 11008, 2048), 0, 215, 248),
    ((1, 3328, 3328, 3328), 1, 82, 96),
])
def test_choice_against_measured_times(choose, shape, b_cm, big, tiles):
    c = choose(*shape, b_cm=b_cm)
    assert c["route"] in ("big", "tiles")
    took = big if c["route"] == "big" else tiles
    assert took <= 1.1 * min(big, tiles), (c, big, tiles)


# ... on the 256 x 256 kernel, the tiles as A is stored, and the tiles on a copy of A
@pytest.mark.parametrize("shape,b_cm,big,tiles,copied", [
    ((8, 2048, 2048, 128), 1, 33, 27, 33),
    ((1, 4096, 4096, 4096), 1, 149, 235, 175),
    ((32, 2048, 2048, 128), 1, 107, 125, 115),
    ((1, 2048, 2048, 2048), 1, 59, 32, 32),
    ((1, 1024, 1024, 1024), 1, 34, 7.5, 13),
    ((1, 563, 6177, 3520), 1, 86, 64, 51),
    ((1, 563, 6177, 3520), 0, 113, 80, 57),
    ((1, 1024, 4096, 4096), 1, 98, 63, 51),
    ((1, 2048, 4096, 4096), 1, 103, 114, 89),
    ((1, 2048, 2048, 4096), 0, 111, 63, 56),
    ((8, 500, 1000, 64), 1, 14, 5.4, 11),
    ((1, 16, 4096, 4096), 1, 92, 11, 17),
    ((7, 964, 5679, 448), 0, 105, 97, 76),
])
def test_choice_for_a_column_major_a(choose, shape, b_cm, big, tiles, copied):
    c = choose(*shape, a_cm=1, b_cm=b_cm)
    took = big if c["route"] == "big" else copied if c["copy_a"] else tiles
    assert took <= 1.1 * min(big, tiles, copied), (c, big, tiles, copied)
    c = choose(*shape, a_cm=1, b_cm=b_cm, copies=0)  # no room: as it is stored
    assert c["route"] == "tiles" and not c["copy_a"] and not c["copy_b"]


def test_consumers_of_the_large_kernel_are_covered(choose):
    """The sizes the consumer test means the 256 x 256 kernel with."""
    assert choose(1, 4090, 4096, 128)["route"] == "big"


def test_small_tiles_do_not_queue_for_lds(choose):
    """[200, 130, 96] . [200, 96, 130]: 3000 tiles of 32 x 64, one ring to a compute unit, take 23.8 us; 64 x 64 take 9."""
    c = choose(200, 130, 130, 96)
    assert c["route"] == "big" or c["kind"] != WAVES


@pytest.mark.parametrize("change", [{"aligned": 0}, {"b_cm": 0, "copies": 1 << 20}])
def test_the_large_kernel_wants_aligned_operands_and_room(choose, change):
    assert choose(1, 4096, 4096, 4096)["route"] == "big"
    assert choose(1, 4096, 4096, 4096, **change)["route"] == "tiles"


@pytest.mark.parametrize("shape,a_cm,b_cm,route", [
    ((1, 4096, 4096, 48), 0, 1, "tiles"),         # k in no whole steps of 32
    ((1, 5, 7, 6), 0, 1, "elements"),             # rows shorter than a chunk
    ((1, 4096, 4096, 0), 0, 1, "elements"),       # an empty sum
    ((2, 4, 49152, 64), 1, 1, "big"),             # rows of A of four elements, tiles enough: a copy
    ((1, 4, 512, 64), 1, 1, "elements"),
    ((1, 16, 64, 1 << 23), 0, 1, "elements"),     # offsets inside a tile past 31 bits
])
def test_what_no_tile_takes(choose, shape, a_cm, b_cm, route):
    assert choose(*shape, a_cm=a_cm, b_cm=b_cm)["route"] == route


def test_ranges_fit_the_scratch_memory(choose):
    assert choose(1, 300, 512, 5504)["ksplit"] > 1
    assert choose(1, 300, 512, 5504, scratch=0)["ksplit"] == 1
    c = choose(1, 300, 512, 5504, scratch=3 * 300 * 512 * 4)
    assert c["ksplit"] <= 3


# ---- two products of one A ---------------------------------------------------------------------
@pytest.fixture(scope="module")
def choose_two(exe):
    def many(shapes):
        """Of (m, n, k, a_cm, b_cm, aligned, scratch, reads_first): what both products are given."""
        lines = "".join(f"1 {m} {n} {k} {a_cm} {b_cm} {aligned} {scratch} {COPIES} {reads_first}\n"
                        for m, n, k, a_cm, b_cm, aligned, scratch, reads_first in shapes)
        out = subprocess.run([str(exe), "two"], input=lines, capture_output=True, text=True, check=True).stdout.splitlines()
        return [dict(zip(("half", "tiles", "kind", "bm", "bn", "ksplit", "us", "one_us"), [int(x) for x in line.split()[:6]] +
                         [float(x) for x in line.split()[6:]])) for line in out]

    return many


def test_two_products_take_the_kernels_their_gpu_test_names(choose_two):
    """... test_gpu_matmul_two.py's shapes: 64 or 128 columns of both, tiles as (kind, k ranges), or none of these."""
    for reads_first in (0, 1):
        got = choose_two([(m, n, k, int(a == COL), int(order == COL), 1, SCRATCH, reads_first) for b, m, n, k, order, a in SHAPES])
        for shape, c, want in zip(SHAPES, got, TAKEN):
            route = c["half"] or ((c["kind"], c["ksplit"]) if c["tiles"] else None)
            assert shape[0] > 1 or route == want[reads_first], (shape, reads_first, c)
    routes = {r for w in TAKEN for r in w}
    assert {64, 128, None} < routes and {r[0] for r in routes if isinstance(r, tuple)} == {STAGED, DIRECT, WAVES}
    assert any(isinstance(r, tuple) and r[1] > 1 for r in routes)


def test_two_products_of_drawn_shapes(choose_two):
    """A second consumer that reads what the first leaves never has tiles of one range (each in a workgroup of its own);
    ranges of both fit the scratch memory; a workgroup of both wants whole stages and chunks; and what is taken is
    expected to be faster than one after the other."""
    rng = random.Random(5)
    near = lambda lo, hi: int(round(lo * (hi / lo) ** rng.random()))  # noqa: E731
    shapes = [(near(1, 1024), rng.choice([1, 1, 8]) * near(1, 700), rng.choice([1, 8, 64]) * near(1, 32), rng.choice([0, 0, 0, 1]), rng.randint(0, 1),
               rng.choice([0, 1, 1]), rng.choice([0, 1 << 20, SCRATCH]), rng.randint(0, 1)) for _ in range(4000)]
    seen = set()
    for (m, n, k, a_cm, b_cm, aligned, scratch, reads_first), c in zip(shapes, choose_two(shapes)):
        what = (m, n, k, a_cm, b_cm, aligned, scratch, reads_first, c)
        if c["half"]:
            assert not a_cm and aligned and k % 64 == 0 and (b_cm or n % 8 == 0), what
        elif c["tiles"]:
            assert c["ksplit"] > 1 or not reads_first, what
            assert c["ksplit"] == 1 or 2 * m * n * 4 * c["ksplit"] <= scratch, what
            assert c["kind"] == STAGED or (not a_cm and aligned and (b_cm or n % 8 == 0) and k % (64 if c["kind"] == DIRECT else 32) == 0), what
        if c["half"] or c["tiles"]:
            assert c["us"] <= 2 * c["one_us"] + 0.01 or c["one_us"] == 0, what  # (0: a product with no tiles of its own)
        seen.add((c["half"], c["tiles"], c["tiles"] and c["ksplit"] > 1))
    assert {(0, 0, 0), (64, 0, 0), (128, 0, 0), (0, 1, False), (0, 1, True)} <= seen
