"""The split-K projection kernel of a decode step's rows (``ops.gemm_rows``) at the edges of its tiles: row counts
around 16, columns past the last whole tile, K of one slice, of a part of a pass and past one pass of 1,024; and which calls
of the serving layer take it."""

from __future__ import annotations

import importlib

import pytest
import torch
import torch.nn.functional as F

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


class _Quantised(torch.Tensor):
    """A weight whose own tensor says nothing of its values (as wrapper subclasses of quantised weights do)."""


def test_calls_outside_the_kernel_stay_linear(gdn, cuda):
    """Rows that start off a 16-byte boundary, widths outside the kernel's, more rows, other dtypes, tensor
    subclasses and products that autograd records are F.linear's, bit for bit; the plain call is the kernel's."""
    serving = importlib.import_module("zonos3-mini_amd.serving")
    announce("few-row projections: the rule")
    gen = torch.Generator().manual_seed(77)
    bf = torch.bfloat16
    r = lambda *s: torch.randn(*s, generator=gen).to(bf).to(cuda)
    M, N, K = 4, 64, 256
    x, w = r(M, K), r(N, K)
    assert serving._takes_few_rows(x, w) and torch.equal(serving._few_rows(x, w), gdn.ops.gemm_rows(x, w))
    off = r(M * K + 1)[1:].view(M, K)  # contiguous, two bytes past a boundary
    off_w = r(N * K + 1)[1:].view(N, K)
    assert off.is_contiguous() and off.data_ptr() % 16 == 2
    for a, b in ((off, w), (x, off_w), (r(M, 192), r(N, 192)), (x, r(60, K)), (r(129, K), w), (x.float(), w.float()),
                 (x, w.as_subclass(_Quantised)), (x, r(K, N).T), (r(M, 2 * K)[:, ::2], w)):
        assert not serving._takes_few_rows(a, b)
        assert torch.equal(serving._few_rows(a, b), F.linear(a, b))
    p = torch.nn.Parameter(w)
    assert serving._few_rows(x, p).requires_grad
    with torch.no_grad():
        assert serving._takes_few_rows(x, p)
    with torch.inference_mode():
        assert serving._takes_few_rows(x, p)


def test_a_decode_step_of_unaligned_rows(gdn, cuda):
    """A serving decode step whose rows start off a 16-byte boundary: the results of the same rows on one, to the
    distance between two orders of the projections' sums."""
    from test_gpu_serving_extend import _pair

    serving = importlib.import_module("zonos3-mini_amd.serving")
    announce("serving decode of unaligned rows")
    layers, gen = _pair(serving, cuda, 256, 4, 5400)
    rows = torch.randn(4, 256, generator=gen).to(torch.bfloat16).to(cuda)
    ys = []
    for (layer, batch), at in zip(layers, (0, 1)):
        layer.enable_graph_decode(torch.arange(4, device=cuda), layer.static_tables(cuda, [4]))
        layer.set_static_mode(True)
        batch.is_decode, batch.padded_size = True, 4
        x = torch.empty(4 * 256 + at, dtype=torch.bfloat16, device=cuda)[at:].view(4, 256)
        x.copy_(rows)
        ys.append(layer.forward(x).float())
        torch.cuda.synchronize()
        assert torch.equal(layer._window[:, 0], rows) and layer._win_len.tolist() == [1] * 4
    # (a step from zero states: a bf16 element of the projection rounded the other way, 2^-8 of it, and the output's own)
    assert float((ys[0] - ys[1]).abs().max() / ys[0].abs().max()) < 2e-2
