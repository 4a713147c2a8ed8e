"""The kernel a kernel-level fp16 matmul is given (csrc/backend/f16_gemm_choice.h), without a device."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
STAGED, DIRECT, WAVES = 0, 1, 2
SCRATCH, COPIES = 64 << 20, 128 << 20  # what a queue has


@pytest.fixture(scope="module")
def choose(tmp_path_factory):
    exe = tmp_path_factory.mktemp("choice") / "gemm_choice"
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-I",
                           os.path.join(ROOT, "attention_superoptimizer_amd", "csrc", "backend"), "-o", str(exe),
                           os.path.join(ROOT, "tests", "cpp", "gemm_choice.cc")])

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
