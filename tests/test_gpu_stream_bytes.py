"""tc_count_stream_bytes: the bytes a default count streams, restated from the
CSR: over 16-bit rows of a graph whose vertices all have an id, and over the
32-bit work lists of a graph that the rows do not suit; and a batch's."""
import numpy as np
import pytest

import tcamd
from graphs import CASES

pytestmark = pytest.mark.gpu


def rows_bytes(rp, col):
    """Every edge goes to the end with the longer row, to its source on a tie;
    it is dropped where a row is empty, or the source owns it as its only entry."""
    d = np.diff(rp.astype(np.int64))
    u, v = np.repeat(np.arange(len(d)), d), col.astype(np.int64)
    keep = (d[u] > 0) & (d[v] > 0) & ((d[v] > d[u]) | (d[u] > 1))
    u, v = u[keep], v[keep]
    pull = d[v] > d[u]
    owner, streamed = np.where(pull, v, u), np.where(pull, u, v)
    unit = 16 * -(-d // 8)
    tasks = np.unique(owner)
    return int((8 + unit[streamed]).sum() + (16 + unit[tasks]).sum())


@pytest.mark.parametrize("case", list(CASES))
@pytest.mark.parametrize("orient", [tcamd.ORIENT_DEGREE, tcamd.ORIENT_ID])
def test_rows(ctx, case, orient):
    g = ctx.graph(*CASES[case]()).orient(orient)
    assert g.count_stream_bytes() == (rows_bytes(*g.csr()), True)
    g.close()


def test_without_rows(ctx):
    g = ctx.graph(*tcamd.gen_er(400_001, 1_600_003, 5)).orient(tcamd.ORIENT_DEGREE)
    assert g.count_stream_bytes() == (g.auto_stream_bytes(), False)
    g.close()


def test_batch(ctx):
    e = np.zeros(0, np.uint32)
    graphs = [(*tcamd.gen_er(n, 12 * n, n), n) for n in (200, 3000)] + [(e, e, 5)]
    want = 0
    for s, d, n in graphs[:2]:
        g = ctx.graph(s, d, n).orient(tcamd.ORIENT_DEGREE)
        want += rows_bytes(*g.csr())
        g.close()
    b = ctx.batch(graphs)
    assert b.stream_bytes() == want
    b.close()
