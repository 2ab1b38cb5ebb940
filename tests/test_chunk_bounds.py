"""What the bounds on the bf16 chunk path's outputs (``gdn_testing.out_errs``) see, on the CPU: mistakes planted in the
chunked statement of the oracle -- the carried state left out of one chunk, the in-chunk part cut to its diagonal 16 x 16
blocks -- fail them on the inputs of the GPU tests, by a wide margin; outputs rounded to bf16 pass."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from gdn_testing import OUT_RMS, OUT_ROW, out_errs
from oracle import gdn_oracle as O


def _outputs(d, g, cu, no_state=(), blocks_only=False):
    """The outputs of ``O.chunked_np`` over packed sequences, without Q S0^T in the chunks that start at the positions
    ``no_state`` of their sequence, or with P's diagonal 16 x 16 blocks alone."""
    q, k, v, g, beta = (O._f64(t)[0] for t in (d["q"], d["k"], d["v"], g, d["beta"]))
    o = np.zeros(v.shape)
    for s, (a, e) in enumerate(zip(cu, cu[1:])):
        for h in range(v.shape[1]):
            hk, S = h // (v.shape[1] // q.shape[1]), O._f64(d["s0"])[s, h]
            for c in range(a, e, O.CHUNK):
                r = slice(c, min(e, c + O.CHUNK))
                G, L = np.cumsum(g[r, h]), r.stop - c
                lower = np.tril(np.ones((L, L)))
                decay = np.exp(np.where(lower > 0, G[:, None] - G[None, :], -np.inf))
                A = beta[r, h][:, None] * decay * np.tril(k[r, hk] @ k[r, hk].T, -1)
                U = np.linalg.solve(np.eye(L) + A, beta[r, h][:, None] * (v[r, h] - np.exp(G)[:, None] * (k[r, hk] @ S.T)))
                P = (q[r, hk] @ k[r, hk].T) * decay
                if blocks_only:
                    P = P * (np.arange(L)[:, None] // 16 == np.arange(L)[None, :] // 16)
                carried = 0.0 if c - a in no_state else np.exp(G)[:, None] * (q[r, hk] @ S.T)
                o[r, h] = q.shape[-1]**-0.5 * (carried + P @ U)
                S = np.exp(G[-1]) * S + U.T @ (np.exp(G[-1] - G)[:, None] * k[r, hk])
    return o


@pytest.mark.parametrize("decay", [1.0, 4.0])
@pytest.mark.parametrize("H", [2, 16])
@pytest.mark.parametrize("lengths", [[64, 1, 63], [65, 128, 129], [192, 193, 256, 0, 2]])
def test_planted_mistakes_of_a_chunk(lengths, H, decay):
    cu, _ = O.chunk_tables(lengths)
    d = O.make_inputs(1, sum(lengths), H, H, 128, 128, seed=900 + H + sum(lengths), dtype=torch.bfloat16,
                      state_std=0.02, n_states=len(lengths))
    g = d["g"] * decay
    ref = _outputs(d, g, cu)
    a, e = cu[0], cu[1]
    want, _ = O.chunked_np(*(t[0, a:e] for t in (d["q"], d["k"], d["v"], g, d["beta"])), 128**-0.5, d["s0"][0])
    assert np.abs(ref[a:e] - want).max() < 1e-12
    rms, row = out_errs(torch.from_numpy(ref).to(torch.bfloat16), ref, cu)
    assert rms < OUT_RMS and row < OUT_ROW
    for start in range(0, max(lengths), O.CHUNK):  # one chunk of each sequence
        assert out_errs(_outputs(d, g, cu, no_state=(start,)), ref, cu)[1] > 2 * OUT_ROW, start
    assert out_errs(_outputs(d, g, cu, blocks_only=True), ref, cu)[1] > 2 * OUT_ROW


@pytest.mark.parametrize("decay", [1.0, 0.05])
@pytest.mark.parametrize("T,H,segment", [(2049, 4, 11), (2111, 1, 11), (2303, 8, 18)])
def test_planted_mistake_of_a_segment(T, H, segment, decay):
    """The state carried into one segment left out of its outputs' first chunk alone."""
    d = O.make_inputs(1, T, H, H, 128, 128, seed=T + H, dtype=torch.bfloat16, state_std=0.02, n_states=1)
    g, cu = d["g"] * decay, [0, T]
    ref = _outputs(d, g, cu)
    for start in range(segment * O.CHUNK, T, segment * O.CHUNK):
        assert out_errs(_outputs(d, g, cu, no_state=(start,)), ref, cu)[1] > 2 * OUT_ROW, start
