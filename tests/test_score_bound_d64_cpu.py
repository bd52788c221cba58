"""The certification bound of the route scorer at head_dim 64 (scores_mfma_kernel<64, NW>, csrc/bb_routes.hip), on the CPU.

Same statement and input kinds as test_score_bound_cpu.py, with the counts of a 64-element dot product: 2 blocks of 32 in
the reference order and 4 slices of 16 on the MFMA path.
"""
import numpy as np
import pytest

import test_score_bound_cpu as base

D = 64


def _weights():
    d = np.arange(D)
    c, t, s = d >> 5, (d & 31) >> 1, d >> 4
    return ((16 - np.maximum(t, 1)) + 1 + (2 - np.maximum(c, 1))).astype(np.float64), (6 - np.maximum(s, 1)).astype(np.float64)


@pytest.mark.parametrize("kind", base.KINDS)
def test_bound_covers_both_orders(kind, monkeypatch):
    monkeypatch.setattr(base, "D", D)
    q, k = base._inputs(kind, 40000, base.KINDS.index(kind))
    p = q.astype(np.float64) * k.astype(np.float64)
    exact, a, slack = p.sum(1), np.abs(p), 1 + 2.0 ** -10
    ref = base._ref_order(q, k)
    wr, wm = _weights()
    assert (np.abs(ref - exact) <= base.U * (a * wr).sum(1) * slack + 1e-30).all(), "reference chain exceeds its part"
    top = (np.abs(q).reshape(-1, 4, 16).max(2).astype(np.float64) * np.abs(k).reshape(-1, 4, 16).max(2)).sum(1)
    for final in ("nearest", "truncate"):
        mf = base._mfma_model(q, k, final)
        mpart = base.U * ((a * wm).sum(1) + 32.0 * top)
        assert (np.abs(mf - exact) <= mpart * slack + 1e-30).all(), f"MFMA model exceeds its part ({final})"
        assert (np.abs(ref - mf) <= base.U * ((a * (wr + wm)).sum(1) + 32.0 * top) * slack + 1e-30).all()
