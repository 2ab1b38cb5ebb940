"""The split-K projection kernel of a decode step's rows (``ops.gemm_rows``) at the edges of its tiles: row counts
around 16, columns past the last whole tile, K of one slice, of a part of a pass and past one pass of 1,024."""

from __future__ import annotations

import pytest
import torch

from gdn_testing import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(1, 2056, 1024), (16, 8, 128), (17, 24, 1152), (33, 2056, 2048), (128, 1024, 512),
                                   (5, 40, 384)])
def test_gemm_rows(gdn, cuda, M, N, K):
    announce(f"gemm_rows {M}x{N}x{K}")
    gen = torch.Generator().manual_seed(M + N + K)
    wide = torch.randn(M, K + 64, generator=gen).to(torch.bfloat16).to(cuda)
    x = wide[:, 64:]  # rows a stride apart
    w = torch.randn(N, K, generator=gen).to(torch.bfloat16).to(cuda)
    y = gdn.ops.gemm_rows(x, w)
    torch.cuda.synchronize()
    ref = x.double() @ w.double().T
    # bf16 rounding of the result (half a step, 2^-9 of it, to the next power of two) and fp32 sums of K products:
    # at most K 2^-24 of the sum of their sizes
    bound = 2.0**-8 * ref.abs() + K * 2.0**-24 * (x.double().abs() @ w.double().abs().T)
    assert bool(((y.double() - ref).abs() <= bound).all())
