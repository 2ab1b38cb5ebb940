"""The fp32 chunk forward in slices (phase 1 of a slice beside the state pass of the one before it): each chunk takes
the same steps in the same order as in two launches, so the outputs are equal bit for bit to those of a call that
returns no final state (which is not sliced), and the final state agrees with the oracle's token loop. Slice counts
2 to 8, a shorter last slice, a partial last chunk, several sequences, the state in place."""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

from gdn_testing import announce, rel_err
from oracle import gdn_oracle as O

pytestmark = pytest.mark.gpu

# as for the fp32 chunk kernels in general: sums of n fp32 products, off by about sqrt(n) 2^-24 of their size
TOL = 2e-5


@pytest.mark.parametrize("D,B,T,Hk,Hv,slices", [(128, 1, 4096, 16, 16, 4), (128, 1, 4033, 8, 8, 2),
                                                (128, 2, 2999, 4, 8, 3), (128, 1, 9580, 2, 4, 3),
                                                (128, 1, 3301, 12, 12, 3), (128, 1, 8192, 16, 16, 8),
                                                (64, 1, 4096, 16, 16, 4), (64, 1, 4095, 4, 8, 2)])
def test_slices_equal_two_launches(gdn, cuda, D, B, T, Hk, Hv, slices):
    announce(f"chunk f32 slices D={D} B={B} T={T} Hv={Hv}")
    assert gdn._native.lib().zgdn_chunk32_slices(D, B, T, Hv) == slices  # (the call is sliced, as often as listed)
    gen = torch.Generator().manual_seed(5 + T)
    q, k = (O.l2norm(torch.randn(B, T, Hk, D, generator=gen)) for _ in range(2))
    v = torch.randn(B, T, Hv, D, generator=gen)
    g, beta = -F.softplus(torch.randn(B, T, Hv, generator=gen)), torch.rand(B, T, Hv, generator=gen)
    s0 = 0.02 * torch.randn(B, Hv, D, D, generator=gen)
    args = [x.to(cuda) for x in (q, k, v, g, beta)]
    st = s0.to(cuda)
    o1, _ = gdn.chunk_fwd(*args, initial_state=st, output_final_state=False)
    for state in (torch.empty_like(st), st):  # (the last one over its own input)
        o2, s2 = gdn.chunk_fwd(*args, initial_state=st, final_state=state)
        assert torch.equal(o1, o2)
    _, s3 = gdn.chunk_fwd(*args, initial_state=s0.to(cuda))
    assert torch.equal(s2, s3)
    z1, _ = gdn.chunk_fwd(*args, output_final_state=False)
    z2, _ = gdn.chunk_fwd(*args)
    assert torch.equal(z1, z2)
    n = min(T, 700)  # the oracle's loop over the first tokens, and the state over the last ones from the kernel's own
    o_ref, _ = O.gated_delta_recurrence(q[:, :n], k[:, :n], v[:, :n], g[:, :n], beta[:, :n], None, s0)
    cut = (T - 1) // 64 * 64
    _, mid = gdn.chunk_fwd(*(x[:, :cut].contiguous() for x in args), initial_state=s0.to(cuda))
    _, s_ref = O.gated_delta_recurrence(q[:, cut:], k[:, cut:], v[:, cut:], g[:, cut:], beta[:, cut:], None, mid.cpu())
    eo, es = rel_err(o1[:, :n], o_ref), rel_err(s3, s_ref)
    print(f"fp32 slices D={D} T={T}: output rel err {eo:.2e}, state rel err {es:.2e}")
    assert eo < TOL and es < TOL, (eo, es)
