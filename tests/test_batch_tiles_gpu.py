"""The one-workgroup batch drain where its layers change shape: one or two
16-record tiles per patch position (batches of 16 and 17, window 1 for the s3
layers too), no output record in a layer (the q columns are skipped), and no
record in it at all (a long dropout window: the s3 layers are skipped),
against the fp64 oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from ssla_hip import events
from test_drain_gpu import compare, hidden_close, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [1, 16, 17, 32])
@pytest.mark.parametrize("window", [1, 4, 64])
def test_batch_tiles(batch, window):
    from ssla_hip import hybrid as H
    n, H2, W2 = 400, 16, 20
    say(batch, window)
    w = events.p1_replica(n, 2, H2, W2)
    w.rec.x[::3], w.rec.y[::3] = 7, 9                 # a dense cell in every batch
    w.rec.x[::11] = W2                                # off the grid
    packed = [H.pack_raw_layer(r) for r in w.layers]
    layers = [O.Layer(p.qvgIn, p.goW, p.input_proj, p.ln_gamma, p.ln_beta) for p in packed]
    st = O.S2S3(layers, H2, W2, window, h_init=w.h_init)
    p2, p3, feat, _ = st.run(w.rec.x, w.rec.y, w.rec.feat1)
    with H.Drain.from_packed(packed, H2, W2, window, h_init=w.h_init) as d:
        (out,), _ = d.drain([events.to_records(w.rec)], batch=batch)
        compare(out, p2, p3, feat, f"batch {batch} window {window}")
        td2, td3 = d.counters(0)
        assert np.array_equal(td2, st.td2) and np.array_equal(td3, st.td3)
        for li in range(4):
            assert hidden_close(d.hidden(0, li), st.H[li]), li
