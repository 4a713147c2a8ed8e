"""fp16 matmuls whose stages go to LDS directly: the tile kernel and the wavefronts-split-k kernel."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b_kc", [0, 1])
@pytest.mark.parametrize("batch,m,n,k", [
    (1, 16, 64, 32),        # one step: three wavefronts without work
    (1, 1, 8, 160),         # the smallest rows, five steps
    (2, 17, 72, 96),        # edges of the 16- and 32-row tiles, a batch
    (1, 100, 1000, 480),    # k in whole steps of 32, not of 64
    (1, 96, 1024, 512),
    (1, 500, 520, 64),      # one stage
    (3, 200, 392, 128),
    (1, 300, 1032, 2048),   # ragged 64 x 64 tiles
    (1, 333, 1048, 5504),   # k ranges
    (1, 1025, 2056, 256),   # wide tiles, more than one to a compute unit
])
def test_direct_matmuls_match_float(rt, abi, batch, m, n, k, b_kc):
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    A = torch.randn(batch, m, k, device="cuda", generator=gen).half()
    B = torch.randn((batch, n, k) if b_kc else (batch, k, n), device="cuda", generator=gen).half()
    C = torch.full((batch, m, n), float("nan"), device="cuda", dtype=torch.float16)
    torch.cuda.synchronize()
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    assert abi.mi355_f16_matmul_layout(p(A), p(B), p(C), batch, m, n, k, 0, b_kc) == 0
    assert abi.mi355_sync() == 0
    Bf = B.float().transpose(1, 2).contiguous() if b_kc else B.float()
    want = torch.bmm(A.float(), Bf)
    assert (C.float() - want).abs().max().item() <= 2e-3 * want.abs().max().item()


def _matmul(abi, A, B, batch, m, n, k, a_cm, b_cm):
    """C on the device, between guard rows that must stay as they are; and the product in float."""
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    C = torch.full((batch * m * n + 128,), -7.0, device="cuda", dtype=torch.float16)
    C[64:-64] = float("nan")
    torch.cuda.synchronize()
    assert abi.mi355_f16_matmul_layout(p(A), p(B), p(C[64:]), batch, m, n, k, a_cm, b_cm) == 0
    assert abi.mi355_sync() == 0
    assert (C[:64] == -7).all() and (C[-64:] == -7).all()
    Af = A.float().transpose(1, 2).contiguous() if a_cm else A.float()
    Bf = B.float().transpose(1, 2).contiguous() if b_cm else B.float()
    return C[64:-64].view(batch, m, n).float(), torch.bmm(Af, Bf)


@pytest.mark.parametrize("b_cm", [0, 1])
@pytest.mark.parametrize("batch,m,n,k", [
    (1, 129, 3336, 3264),  # 64 x 128 tiles of eight wavefronts in k ranges: a row and eight columns over
    (1, 300, 5504, 2048),  # one range
    (4, 166, 2616, 1024),
    (2, 191, 3272, 1216),  # a row short of a tile, 19 stages
])
def test_wide_tiles_in_one_round(rt, abi, batch, m, n, k, b_cm):
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    A = torch.randn(batch, m, k, device="cuda", generator=gen).half()
    B = torch.randn((batch, n, k) if b_cm else (batch, k, n), device="cuda", generator=gen).half()
    got, want = _matmul(abi, A, B, batch, m, n, k, 0, b_cm)
    # a rounding to fp16, and a sum of k products in fp32: at most k roundings of partial sums of about sqrt(k)
    assert (got - want).abs().max().item() <= 2**-11 * want.abs().max().item() + 2 * k * 2**-24 * k**0.5


@pytest.mark.parametrize("batch,m,n,k,a_cm,b_cm", [
    (32, 500, 1000, 32, 0, 1),    # one step of the 256 x 256 kernel, ragged tiles
    (1, 4090, 4096, 64, 0, 1),    # two
    (1, 4096, 4093, 96, 0, 1),    # three, rows of C on no boundary
    (8, 2048, 2040, 160, 0, 1),   # five: one more than its ring has slots
    (1, 3071, 4099, 224, 0, 1),
    (4, 2048, 2048, 128, 1, 1),   # copies of the operands stored the other way round
    (1, 4096, 4096, 1024, 0, 0),
    (200, 130, 130, 96, 0, 1),    # many ragged tiles, a step left over
    (12, 1040, 1040, 128, 0, 1),
    (1, 563, 6177, 3520, 1, 0),   # a copy of A alone
    (1, 1024, 4104, 4096, 1, 1),
    (7, 964, 1679, 448, 1, 0),
    (2, 4, 512, 64, 1, 1),        # rows of A shorter than a chunk
])
def test_products_of_many_large_tiles(rt, abi, batch, m, n, k, a_cm, b_cm):
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    A = torch.randn((batch, k, m) if a_cm else (batch, m, k), device="cuda", generator=gen).half()
    B = torch.randn((batch, n, k) if b_cm else (batch, k, n), device="cuda", generator=gen).half()
    got, want = _matmul(abi, A, B, batch, m, n, k, a_cm, b_cm)
    # half an fp16 place of the result, and k fp32 additions in another order
    assert ((got - want).abs() <= 2.0 ** -11 * want.abs() + 1e-6 * k ** 0.5 * want.abs().max() + 1e-6).all()


@pytest.mark.parametrize("a_cm,b_cm", [(0, 1), (0, 0), (1, 1), (1, 0)])
@pytest.mark.parametrize("batch,m,n,k", [
    (1, 16, 64, 64), (2, 33, 72, 128), (1, 300, 520, 512), (1, 64, 256, 4096), (1, 3000, 4096, 64), (2, 9, 7, 40)])
@pytest.mark.parametrize("off", [(1, 0, 0), (0, 3, 0), (0, 0, 1), (5, 7, 3)])
def test_operands_on_no_boundary(rt, abi, batch, m, n, k, a_cm, b_cm, off):
    """Bases that are whole elements and nothing more: the kernels of 16-byte chunks leave these to others."""
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    make = lambda count, o: torch.randn(count + 8, device="cuda", generator=gen).half()[o:o + count]  # noqa: E731
    A, B = make(batch * m * k, off[0]), make(batch * n * k, off[1])
    C = torch.full((batch * m * n + 64,), -7.0, device="cuda", dtype=torch.float16)
    out = C[32 + off[2]:32 + off[2] + batch * m * n]
    out.fill_(float("nan"))
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    torch.cuda.synchronize()
    assert abi.mi355_f16_matmul_layout(p(A), p(B), p(out), batch, m, n, k, a_cm, b_cm) == 0
    assert abi.mi355_sync() == 0
    assert (C[:32 + off[2]] == -7).all() and (C[32 + off[2] + batch * m * n:] == -7).all()
    Af = A.view(batch, k, m).float().transpose(1, 2).contiguous() if a_cm else A.view(batch, m, k).float()
    Bf = B.view(batch, n, k).float().transpose(1, 2).contiguous() if b_cm else B.view(batch, k, n).float()
    want = torch.bmm(Af, Bf)
    # half an fp16 place of the result, and k fp32 additions in another order
    assert ((out.view(batch, m, n).float() - want).abs() <= 2.0 ** -11 * want.abs() + 1e-6 * k ** 0.5 * want.abs().max() + 1e-6).all()
