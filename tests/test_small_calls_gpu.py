"""Small whole-ring calls (k_small_order) at the sizes where the ordering takes
another route, against the oracle: one record per thread of the one-launch
ordering (1024), the records its LDS holds (8192), more of either, and the
number of grid cells it has threads for (1024, over several blocks).  Off-grid
records, an empty block and nonzero counters before the call are part of each.
"""
import numpy as np
import pytest

from oracle import oracle as O
from ssla_hip import events
from test_drain_gpu import compare, hidden_close, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def H():
    from ssla_hip import hybrid, lib
    lib.load()
    lib.check_layout()
    return hybrid


def _drain(H, H2, W2, counts, window):
    """Two calls in a row, so that the second finds counters and state."""
    w = events.p1_replica(max(2 * max(counts), 64), 3, H2, W2)
    packed = [H.pack_raw_layer(r) for r in w.layers]
    layers = [O.Layer(p.qvgIn, p.goW, p.input_proj, p.ln_gamma, p.ln_beta) for p in packed]
    nb = len(counts)
    say(H2, W2, counts, window)
    with H.Drain.from_packed(packed, H2, W2, window, n_blocks=nb, h_init=w.h_init) as d:
        states = [O.S2S3(layers, H2, W2, window, h_init=w.h_init) for _ in range(nb)]
        for call in range(2):
            recs = []
            for b, n in enumerate(counts):
                o = (b + call) % 2
                r = events.Records(w.rec.t[o:o + n], w.rec.x[o:o + n].copy(), w.rec.y[o:o + n].copy(),
                                   w.rec.feat1[o:o + n])
                r.x[5::13] = W2                            # off the grid
                recs.append(r)
            outs, _ = d.drain([events.to_records(r) for r in recs])
            for b, r in enumerate(recs):
                if not r.x.size:
                    continue
                p2, p3, feat, _ = states[b].run(r.x, r.y, r.feat1)
                compare(outs[b], p2, p3, feat, f"call {call} block {b}")
        for b, n in enumerate(counts):
            td2, td3 = d.counters(b)
            assert np.array_equal(td2, states[b].td2) and np.array_equal(td3, states[b].td3)
            for li in range(4):
                assert hidden_close(d.hidden(b, li), states[b].H[li]), (b, li)


@pytest.mark.parametrize("n", [1, 63, 1023, 1024, 1025, 8192, 8193])
def test_record_counts(H, n):
    _drain(H, 16, 20, [n], 4)


@pytest.mark.parametrize("H2,W2,counts", [
    (32, 32, [1000]),                      # 1024 cells in one block
    (16, 16, [300, 0, 17, 500]),           # 1024 cells in four, one empty
    (16, 16, [1000, 900, 1, 800]),         # past one record per thread
    (32, 34, [700]),                       # 1088 cells: the larger call's route
])
def test_cells_and_blocks(H, H2, W2, counts):
    _drain(H, H2, W2, counts, 2)
