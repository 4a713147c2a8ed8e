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
