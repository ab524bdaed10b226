"""Per-vertex counts of a graph that is oriented anew: the task lists of the
kernel over the CSR are those of the new orientation.  The graph is one that
16-bit list rows do not suit: more than 65,535 vertices, short lists, and too
few entries among the 65,535 vertices of largest degree."""
import numpy as np
import pytest

import oracle as orc
import tcamd

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def records():
    n, m = 600_000, 1_200_000
    s, d = tcamd.gen_er(n, m, 5)
    # one vertex joined to 3,000 and one to 300: under ID out-degrees that the
    # degree orientation has nowhere
    s = np.concatenate([s, np.full(3000, n), np.full(300, n + 1)]).astype(np.uint32)
    d = np.concatenate([d, np.arange(3000) * 200, np.arange(300) * 2000]).astype(np.uint32)
    deg = np.bincount(s, minlength=n + 2) + np.bincount(d, minlength=n + 2)
    assert np.sort(deg)[-65535:].sum() < 0.85 * len(s)  # a bound on the entries with an id
    return s, d


def test_counts_follow_the_orientation(ctx, records):
    s, d = records
    g = ctx.graph(s, d)
    widest = []
    for o in (tcamd.ORIENT_DEGREE, tcamd.ORIENT_ID, tcamd.ORIENT_ADIR, tcamd.ORIENT_ID):
        g.orient(o)
        i = g.info()
        assert i.sum_in_out < 32 * i.m_oriented
        widest.append(i.max_out_degree)
        rp, col = g.csr()
        for _ in range(3):
            np.testing.assert_array_equal(g.count_per_vertex(), orc.count_per_vertex(rp, col))
    assert min(widest) <= 64 and max(widest) > 2048
    g.close()
