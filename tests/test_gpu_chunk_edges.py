"""The bf16 chunk kernels at the edges of the state pass's loops (1, 2, 3 and 4 chunks, full and partial last ones) in
both of its forms -- one value block a workgroup with output waves (few chains), two blocks without (many) -- and
under decays so strong that a chunk's total decay leaves fp32's range (the outputs' products must not pass through
factors like exp(G_i - G_L)). Tolerances of the bf16 path: outputs within the bounds of ``gdn_testing.out_errs``, which
tests/test_chunk_bounds.py shows to see a missing term of one chunk on these inputs, states 1e-3 relative."""

from __future__ import annotations

import pytest
import torch

from gdn_testing import OUT_RMS, OUT_ROW, announce, out_errs, rel_err
from oracle import gdn_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("decay", [1.0, 4.0])
@pytest.mark.parametrize("H", [2, 16])
@pytest.mark.parametrize("lengths", [[64, 1, 63], [65, 128, 129], [192, 193, 256, 0, 2]])
def test_chunk_counts_and_strong_decay(gdn, cuda, lengths, H, decay):
    announce(f"chunk edges {lengths} H={H} decay x{decay}")
    cu, _ = O.chunk_tables(lengths)
    d = O.make_inputs(1, sum(lengths), H, H, 128, 128, seed=900 + H + sum(lengths), dtype=torch.bfloat16,
                      state_std=0.02, n_states=len(lengths))
    g = d["g"] * decay  # about -0.8 a token: a chunk's G_L about -52, times 4 about -206 (exp(103) overflows)
    o, s = gdn.chunk_fwd(*(t.to(cuda) for t in (d["q"], d["k"], d["v"], g, d["beta"])), initial_state=d["s0"].to(cuda),
                         cu_seqlens=torch.tensor(cu, dtype=torch.int32, device=cuda))
    torch.cuda.synchronize()
    o_ref, s_ref = O.gated_delta_recurrence(d["q"], d["k"], d["v"], g, d["beta"], None, d["s0"], cu_seqlens=cu)
    rms, row = out_errs(o, o_ref, cu)
    print(f"[errors] rms {rms:.3e}, row {row:.3e}, state {rel_err(s, s_ref):.3e}")
    assert rms < OUT_RMS and row < OUT_ROW and rel_err(s, s_ref) < 1e-3, (rms, row, rel_err(s, s_ref))


@pytest.mark.parametrize("decay", [1.0, 0.05])
@pytest.mark.parametrize("T,H,segmented", [(2048, 4, False), (2049, 4, True), (2111, 1, True), (2433, 4, True),
                                           (2240, 8, False), (2303, 8, True)])
def test_plain_and_segmented_around_the_plan_line(gdn, cuda, T, H, segmented, decay):
    """Prompts around the length from which the state pass is cut into segments (33 chunks of up to 4 heads, 36 of 8),
    partial last chunks and last segments included: each takes the form that the plan says and meets the bounds of the
    path, also where the decay is so slow (-0.04 a token) that the state carried into a segment is most of the outputs
    of its first rows."""
    announce(f"chunk plan line T={T} H={H} decay x{decay}")
    assert (int(gdn._native.lib().zgdn_chunk_segment_workspace_size(1, T, H)) > 0) == segmented
    d = O.make_inputs(1, T, H, H, 128, 128, seed=T + H, dtype=torch.bfloat16, state_std=0.02, n_states=1)
    g = d["g"] * decay
    o, s = gdn.chunk_fwd(*(t.to(cuda) for t in (d["q"], d["k"], d["v"], g, d["beta"])), initial_state=d["s0"].to(cuda))
    torch.cuda.synchronize()
    o_ref, s_ref = O.gated_delta_recurrence(d["q"], d["k"], d["v"], g, d["beta"], None, d["s0"])
    rms, row = out_errs(o, o_ref)
    print(f"[errors] rms {rms:.3e}, row {row:.3e}, state {rel_err(s, s_ref):.3e}")
    assert rms < OUT_RMS and row < OUT_ROW and rel_err(s, s_ref) < 1e-3, (rms, row, rel_err(s, s_ref))
