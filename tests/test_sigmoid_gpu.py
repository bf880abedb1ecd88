"""The gate of a strongly negative g: sigmoid(g) is subnormal in fp32 from
g = -87.34 to g = -88.72, and still scales a large state.

One record, q and v rows of L4 zero, its g rows g times the record's first
feature (1): the nine cells of its patch go from h to sigmoid(g) h.  The
exponential's argument g log2(e) is rounded to 2^-18 (127 has 17 fraction bits),
2.7e-6 of the result, and a subnormal sigmoid to 1.4e-45, 2e-7 of it: 1e-5.
"""
import numpy as np
import pytest

from ssla_hip import events
from test_drain_gpu import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,group", [(0, 0), (8, 0), (8, 6)])
@pytest.mark.parametrize("g", [-20.0, -87.0, -87.5, -88.0, -88.5])
def test_subnormal_gate(batch, group, g):
    from ssla_hip import hybrid as H
    say("sigmoid", g, batch, group)
    H2, W2 = 16, 20
    w = events.p1_replica(64, 3, H2, W2)
    packed = [H.pack_raw_layer(r) for r in w.layers]
    q = packed[0].qvgIn
    q[:] = 0
    q[:, 2 * q.shape[1] // 3:, 0] = g
    rec = events.to_records(w.rec)[:1].copy()
    rec["x"], rec["y"], rec["feat1"] = 10, 8, 0
    rec["feat1"][0, 0] = 1
    h0 = np.float32(1e38) if g < -80 else np.float32(1)
    with H.Drain.from_packed(packed, H2, W2, 4, h_init=w.h_init) as d:
        d.set_hidden(0, 0, np.full_like(d.hidden(0, 0), h0))
        d.drain([rec], batch=batch, group=group)
        h = d.hidden(0, 0)
    cy, cx = np.divmod(np.arange(H2 * W2), W2)
    near = (np.abs(cx - 10) <= 1) & (np.abs(cy - 8) <= 1)
    want = float(h0) / (1 + np.exp(-g))
    assert np.all(h[~near] == h0)
    assert np.all(np.abs(h[near] - want) <= 1e-5 * want), (h[near].min(), h[near].max(), want)
