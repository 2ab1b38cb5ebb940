"""The fp32 chunk kernels where their work split can go wrong: more phase-1 items than CUs (a workgroup walks
several items, the next one's rows loaded during the last), chunk counts of 1, 2, 3 and more (the state pass's
two operand buffers), partial last chunks, bf16 gate inputs, against the oracle's token loop."""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

from gdn_testing import announce, rel_err
from oracle import gdn_oracle as O

pytestmark = pytest.mark.gpu

# Both kernels and the oracle hold everything in fp32 or better; a sum of n products of rounded terms is off by
# about sqrt(n) 2^-24 of its size, the chain of 64-token inverses and 11 chunks adds such terms: a few 1e-6, and
# max |err| / max |ref| of heavy-tailed outputs some times that.
TOL = 2e-5


@pytest.mark.parametrize("D,Hk,Hv,gate", [(64, 8, 16, False), (128, 16, 16, False), (128, 8, 16, True)])
def test_many_items_ragged(gdn, cuda, D, Hk, Hv, gate):
    lengths = [700, 65, 1, 128, 191, 64, 449]  # 11, 2, 1, 2, 3, 1, 8 chunks: 448 items at 16 heads
    cu, _ = O.chunk_tables(lengths)
    announce(f"chunk f32 items D={D} Hk={Hk} Hv={Hv} gate={gate}")
    T, n = sum(lengths), len(lengths)
    gen = torch.Generator().manual_seed(41 + D + Hk)
    q, k = (torch.randn(1, T, Hk, D, generator=gen) for _ in range(2))
    v = torch.randn(1, T, Hv, D, generator=gen)
    a, b = (torch.randn(1, T, Hv, generator=gen) for _ in range(2))
    s0 = 0.02 * torch.randn(n, Hv, D, D, generator=gen)
    kw = {}
    if gate:  # raw rows, bf16 gate inputs
        a, b = a.bfloat16(), b.bfloat16()
        A_log, dt_bias = 0.3 * torch.randn(Hv, generator=gen), 0.3 * torch.randn(Hv, generator=gen)
        kw = dict(A_log=A_log.to(cuda), dt_bias=dt_bias.to(cuda), use_qk_l2norm=True, beta_is_logit=True)
        qr, kr = O.l2norm(q), O.l2norm(k)
        g, beta = -A_log.exp() * F.softplus(a.float() + dt_bias), b.float().sigmoid()
        ga, gb = a, b
    else:
        q, k = O.l2norm(q), O.l2norm(k)
        qr, kr = q, k
        g, beta = -F.softplus(a), b.sigmoid()
        ga, gb = g, beta
    o, s = gdn.chunk_fwd(q.to(cuda), k.to(cuda), v.to(cuda), ga.to(cuda), gb.to(cuda), initial_state=s0.to(cuda),
                         cu_seqlens=torch.tensor(cu, dtype=torch.int32, device=cuda), **kw)
    torch.cuda.synchronize()
    o_ref, s_ref = O.gated_delta_recurrence(qr, kr, v, g, beta, None, s0, cu_seqlens=cu)
    eo, es = rel_err(o, o_ref), rel_err(s, s_ref)
    print(f"fp32 items D={D}: output rel err {eo:.2e}, state rel err {es:.2e}")
    assert eo < TOL and es < TOL, (eo, es)


@pytest.mark.parametrize("D,dtype,far_gates", [(128, torch.float32, False), (128, torch.float32, True),
                                               (64, torch.bfloat16, True), (64, torch.float32, False)])
def test_rows_far_apart(gdn, cuda, D, dtype, far_gates):
    """Rows 64 MiB apart (a chunk of them is past 4 GiB) give the results of dense rows, bit for bit."""
    announce(f"chunk f32 rows far apart D={D} {dtype} gates {far_gates}")
    T, H = 65, 2
    gen = torch.Generator(device=cuda).manual_seed(43 + D)
    q, k, v = (torch.randn(1, T, H, D, generator=gen, device=cuda).to(dtype) for _ in range(3))
    g = -torch.rand(1, T, H, generator=gen, device=cuda).to(dtype)
    beta = torch.rand(1, T, H, generator=gen, device=cuda).to(dtype)
    ld = 2**26 // dtype.itemsize + 64
    buf = torch.empty(T * ld, dtype=dtype, device=cuda).view(T, ld)

    def far(x, col):
        view = buf[:, col:col + x[0, 0].numel()].view(1, *x.shape[1:])
        view.copy_(x)
        return view

    wide = [far(x, 512 * i) for i, x in enumerate((q, k, v))]
    gates = [far(x, 512 * i + 256 + 8) for i, x in enumerate((g, beta))] if far_gates else [g, beta]
    o, s = gdn.chunk_fwd(*wide, *gates, use_qk_l2norm=True)
    o_ref, s_ref = gdn.chunk_fwd(q, k, v, g, beta, use_qk_l2norm=True)
    assert wide[0].stride(1) == ld and bool(o_ref.any())
    assert torch.equal(o, o_ref) and torch.equal(s, s_ref)
