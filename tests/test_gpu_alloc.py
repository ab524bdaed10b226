"""Pooled device memory and staged uploads: records come back as they went in
at the borders of the staged path and its 4 MiB chunks, and contexts that come,
go and work side by side on threads count what the oracle counts."""
import threading

import numpy as np
import pytest

import oracle as orc
import tcamd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [2 ** 21 - 1, 2 ** 21, 2 ** 21 + 1, 3 * 2 ** 20 + 7, 9 * 2 ** 20 + 3])
def test_upload_round_trip(ctx, m):
    r = np.random.default_rng(m)
    s, d = (r.integers(0, 1 << 20, m, dtype=np.uint32) for _ in range(2))
    g = ctx.graph(s, d)
    gs, gd = g.edges()
    assert np.array_equal(gs, s) and np.array_equal(gd, d)
    g.close()


def test_contexts_on_threads():
    sizes = [(3000, 20000), (700, 60000), (70000, 900000), (200000, 2100000)]
    graphs = [tcamd.gen_er(n, m, n) for n, m in sizes]
    expect = [orc.pipeline_count(s, d, "degree")[0] for s, d in graphs]
    bad = []

    def work(k):
        for r in range(3):  # blocks pass from context to context
            with tcamd.Context(0) as c:
                for i in np.random.default_rng(10 * k + r).permutation(len(graphs)):
                    g = c.graph(*graphs[i])
                    for o in (tcamd.ORIENT_DEGREE, tcamd.ORIENT_ADIR):
                        g.orient(o)
                        if g.count().count != expect[i]:
                            bad.append((k, r, i, o))
                    if i % 2:
                        g.close()

    ts = [threading.Thread(target=work, args=(k,)) for k in range(3)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not bad
