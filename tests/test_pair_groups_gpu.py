"""Projection + recurrence over groups of pairs (k_pscan) at the sizes where
a group's shape changes, against the fp64 oracle.

The pairs of a cell form groups of kGP = 176 of their own when there are
more than kGW = 88 of them; smaller cells share a group.  A group's pairs are
dealt into 16-pair tiles per patch position.  The same code runs at s2 (every
record) and at s3 (every fourth record of a cell at window 4).
"""
import numpy as np
import pytest

from oracle import oracle as O
from ssla_hip import events
from test_drain_gpu import compare, hidden_close, p1_setup, say

pytestmark = pytest.mark.gpu

GP, GW = 176, 88


@pytest.fixture(scope="module")
def H():
    from ssla_hip import hybrid, lib
    lib.load()
    lib.check_layout()
    return hybrid


def _check(H, n, x, y, tag):
    say(tag, n)
    w, d, layers = p1_setup(H, n)
    w.rec.x[:], w.rec.y[:] = x, y
    with d:
        (out,), _ = d.drain([events.to_records(w.rec)])
        st = O.S2S3(layers, w.H2, w.W2, 4, h_init=w.h_init)
        p2, p3, feat, _ = st.run(w.rec.x, w.rec.y, w.rec.feat1)
        compare(out, p2, p3, feat, tag)
        for li in range(4):
            assert hidden_close(d.hidden(0, li), st.H[li]), li


@pytest.mark.parametrize("n", [1, 16, 17, GW, GW + 1, GP, GP + 1, 4 * GW + 1, 2 * GP + 1,
                               4 * GP + 1, 10 * GP - 1])
def test_one_centre_cell(H, n):
    """Nine cells of n pairs each at s2, of about n / 4 at s3: a lone group, a
    full one, full ones and a remainder of one pair."""
    _check(H, n, 10, 8, f"one_cell_{n}")


@pytest.mark.parametrize("n,cells", [(320, 320), (500, 40), (3000, 12)])
def test_shared_groups(H, n, cells):
    """Cells of one to a few hundred pairs in ring orders that interleave
    them: groups of many cells, and shared groups next to cells with groups
    of their own; border cells have fewer patch positions."""
    r = np.random.default_rng(n)
    c = r.permutation(320)[:cells][r.integers(0, cells, n)] if cells < 320 else r.permutation(320)
    _check(H, n, c % 20, c // 20, f"shared_{n}_{cells}")


def test_more_groups_than_the_key_scan_holds(H):
    """Past 6144 groups a cell (1.08 M records) the group list is built by the
    wide launches: one call equals the same ring in two."""
    n = 6144 * GP
    w, d, _ = p1_setup(H, 20_000)
    recs = np.tile(events.to_records(w.rec), n // 20_000 + 1)[:n]
    say("wide group list", n)
    with d:
        (a,), _ = d.drain([recs])
        ha = [d.hidden(0, li) for li in range(4)]
    w, d, _ = p1_setup(H, 20_000)
    with d:
        (b0,), _ = d.drain([recs[:n // 2]])
        (b1,), _ = d.drain([recs[n // 2:]])
        hb = [d.hidden(0, li) for li in range(4)]
    b = np.concatenate([b0, b1])
    assert np.array_equal(a["pass2"], b["pass2"]) and np.array_equal(a["pass3"], b["pass3"])
    # the group boundaries move: the same sums in another association, about
    # 1e-6 of |h| over a run, as between the drain and its oracle
    assert all(hidden_close(x, y) for x, y in zip(ha, hb))
    assert np.abs(a["s3_feat"] - b["s3_feat"]).max() <= 1e-4
