"""Non-finite features and states stay where the recurrence takes them: in the
3 x 3 cells of the records that carry them.

Cells of few pairs share a group of the projection + recurrence kernel, across
blocks too (keys run block by block), so a cell's run begins in the middle of a
group, behind another cell's.  Everything outside the poisoned neighbourhood
equals a run without the poison bit for bit: the same records in the same
groups, with the same sums.
"""
import numpy as np
import pytest

from ssla_hip import events
from test_drain_gpu import say

pytestmark = pytest.mark.gpu

H2, W2 = 16, 20


@pytest.fixture(scope="module")
def H():
    from ssla_hip import hybrid, lib
    lib.load()
    lib.check_layout()
    return hybrid


def _near(li, x, y):
    """Cells of layer li's grid within the 3 x 3 patch of s2 cell (x, y)."""
    s = 0 if li < 2 else 1
    h, w = H2 >> s, W2 >> s
    cy, cx = np.divmod(np.arange(h * w), w)
    return (np.abs(cx - (x >> s)) <= 1) & (np.abs(cy - (y >> s)) <= 1)


def _run(H, n, nb, poison, state):
    """Two calls with records at (2, 2) of block 0 (poisoned) and at (17, 13)
    of the last block.  poison: feature value of one record of the first call;
    state: value of the stored states around (2, 2) before it."""
    w = events.p1_replica(max(8 * n, 64), 3, H2, W2)
    packed = [H.pack_raw_layer(r) for r in w.layers]
    outs, t = [], events.to_records(w.rec)
    with H.Drain.from_packed(packed, H2, W2, 1, n_blocks=nb, h_init=w.h_init) as d:
        if state is not None:
            for li in range(4):
                h = d.hidden(0, li)
                h[_near(li, 2, 2)] = state
                d.set_hidden(0, li, h)
        for call in range(2):
            a, b = t[2 * call * n:(2 * call + 1) * n].copy(), t[(2 * call + 1) * n:(2 * call + 2) * n].copy()
            a["x"], a["y"], b["x"], b["y"] = 2, 2, 17, 13
            if poison is not None and call == 0:
                a["feat1"][n // 2, 5] = poison
            (o, *rest), _ = d.drain([np.concatenate([a, b])] if nb == 1 else [a, b])
            outs.append(o[n:] if nb == 1 else rest[0])
        hid = [[d.hidden(b, li) for li in range(4)] for b in range(nb)]
    return outs, hid


@pytest.mark.parametrize("poison,state", [(np.inf, None), (np.nan, None), (None, -np.inf),
                                          (None, np.nan)])
@pytest.mark.parametrize("nb", [1, 2])
@pytest.mark.parametrize("n", [1, 7, 25, 44, 200])
def test_poison_stays_in_its_cells(H, n, nb, poison, state):
    say("nonfinite", n, nb, poison, state)
    clean, ch = _run(H, n, nb, None, None)
    got, gh = _run(H, n, nb, poison, state)
    for a, b in zip(clean, got):
        for f in ("pass2", "pass3", "s3_feat"):
            assert np.array_equal(a[f], b[f]), f
    for b in range(nb):
        for li in range(4):
            far = ~_near(li, 2, 2) if b == 0 else np.ones(len(gh[b][li]), bool)
            assert np.array_equal(gh[b][li][far], ch[b][li][far]), (b, li)
    # (an infinite state times a sigmoid of zero is NaN: either way not finite)
    assert not np.isfinite(gh[0][0][_near(0, 2, 2)]).all()
