"""AUTO over the 16-bit list layer: rows at the borders of 16-byte units,
128-byte lines and the 64-unit own-row load, work lists across the 64-entry
refills, the 65,535-id border and graphs with a tail, against closed forms,
the oracle and the 32-bit tasks (explicit thresholds keep a count there)."""
import numpy as np
import pytest

import oracle as orc
import tcamd
from graphs import rmat
from tcamd import learned

pytestmark = pytest.mark.gpu

ORIENTS = (tcamd.ORIENT_ID, tcamd.ORIENT_DEGREE, tcamd.ORIENT_ADIR, tcamd.ORIENT_KCORE,
           tcamd.ORIENT_DEGREE_TRICORE, tcamd.ORIENT_DEGENERACY)


def complete(n):
    u, v = np.triu_indices(n, 1)
    return u.astype(np.uint32), v.astype(np.uint32)


def check(ctx, s, d, expect=None, n=0, orients=ORIENTS):
    for o in orients:
        g = ctx.graph(s, d, n).orient(o)
        want = g.count(auto_thresholds=[64, 2048, 0, 8]).count if expect is None else expect
        assert g.count().count == want
        assert g.count(grid_size=3).count == want
        g.close()


@pytest.mark.parametrize("n", [62, 65, 72, 73, 129, 130, 256, 257, 513, 514, 1030])
def test_complete_graphs(ctx, n):
    check(ctx, *complete(n), expect=n * (n - 1) * (n - 2) // 6)


@pytest.mark.parametrize("n", [65534, 65535, 65536, 65537, 70001])
def test_id_border(ctx, n):
    s, d = tcamd.gen_er(n, 2_000_003, 7)
    # the dense part reaches the last ids and lifts the average list
    hs, hd = complete(300)
    perm = np.concatenate([np.arange(n - 150, n), np.arange(150)]).astype(np.uint32)
    s, d = np.concatenate([s, perm[hs]]), np.concatenate([d, perm[hd]])
    expect = orc.pipeline_count(s, d, "degree")[0]
    check(ctx, s, d, expect, n, (tcamd.ORIENT_ID, tcamd.ORIENT_DEGREE, tcamd.ORIENT_ADIR))


@pytest.mark.parametrize("scale,ef", [(8, 24), (12, 16), (16, 16), (17, 8), (18, 16)])
def test_skewed_with_and_without_tail(ctx, scale, ef):
    s, d = rmat(scale, ef, scale)
    check(ctx, s, d)
    p = np.random.default_rng(scale).permutation(1 << scale).astype(np.uint32)
    check(ctx, p[s], p[d], orients=(tcamd.ORIENT_ID, tcamd.ORIENT_ADIR))


def test_learned_count_and_many_lists(ctx):
    # a hub that meets every list of a 20,000-vertex graph: work lists far
    # beyond one refill of the bounds ring
    s, d = tcamd.gen_er(20000, 500_000, 3)
    hub = np.arange(1, 20000, dtype=np.uint32)
    s, d = np.concatenate([s, np.zeros_like(hub)]), np.concatenate([d, hub])
    expect = orc.pipeline_count(s, d, "degree")[0]
    check(ctx, s, d, expect)
    g = ctx.graph(s, d).orient(tcamd.ORIENT_ADIR)
    assert g.count_learned(learned.load(ctx)).count == expect
    assert g.count_learned(None).count == expect
    g.close()


@pytest.mark.parametrize("n", [65534, 65535, 65536])
def test_batch_id_border(ctx, n):
    """Graphs up to 65,535 vertices take 16-bit local ids; one more vertex in
    any of them sends the batch to the 32-bit tasks."""
    e = np.zeros(0, np.uint32)
    s, d = tcamd.gen_er(n, 400_003, 11)
    last = (np.array([0, n - 1, n - 1], np.uint32), np.array([n - 1, 1, 0], np.uint32), n)
    graphs = [(*complete(70), 70), (e, e, 3), (s, d, n), (*complete(9), 64), last,
              (*complete(513), 600), (e, e, 1)]
    expect = [orc.pipeline_count(a, b, "degree")[0] if len(a) else 0 for a, b, _ in graphs]
    b = ctx.batch(graphs)
    for sched in (None, dict(grid=3), dict(form=1)):
        for _ in range(3):  # replays of the captured launch
            assert b.count(sched)[0].tolist() == expect
    assert b.count_pergraph()[0].tolist() == expect
    b.close()


@pytest.mark.parametrize("make,n", [(lambda: complete(130), 0), (lambda: rmat(12, 16, 5), 4096),
                                    (lambda: rmat(17, 12, 6), 1 << 17)])
def test_per_vertex(ctx, make, n):
    """Every entry against the oracle's, before and after a plain count of the
    same graph (which builds the layer without the credits)."""
    s, d = make()
    for o in (tcamd.ORIENT_ID, tcamd.ORIENT_ADIR):
        g = ctx.graph(s, d, n).orient(o)
        want = orc.count_per_vertex(*g.csr())
        assert g.count().count == want.sum()
        for _ in range(2):
            np.testing.assert_array_equal(g.count_per_vertex(), want)
        assert g.count().count == want.sum()
        g.close()


@pytest.mark.parametrize("blocks", [1, 977, 30000])
@pytest.mark.parametrize("make,n", [(lambda: rmat(17, 8, 3), 1 << 17),        # 16-bit rows and a tail
                                    (lambda: tcamd.gen_er(70001, 300_007, 5), 0),  # over 65,535 ids
                                    (lambda: tcamd.gen_er(300_001, 900_001, 5), 0),  # 32-bit rows
                                    (lambda: complete(1030), 0)])                  # long rows, no tail
def test_hu(ctx, make, n, blocks):
    s, d = make()
    for o in (tcamd.ORIENT_ID, tcamd.ORIENT_DEGREE):
        g = ctx.graph(s, d, n).orient(o)
        want = g.count(auto_thresholds=[64, 2048, 0, 8]).count
        for _ in range(2):
            assert g.count("hu", grid_size=blocks).count == want
        g.close()


@pytest.mark.parametrize("kernel", ["bisson", "tricore", "fox"])
@pytest.mark.parametrize("make,n", [(lambda: rmat(17, 16, 3), 1 << 17),               # 16-bit rows, tail
                                    (lambda: tcamd.gen_er(400_001, 1_600_003, 5), 0),  # 32-bit rows
                                    (lambda: complete(1800), 0)])                  # no tail, long rows
def test_bisson_tricore_fox(ctx, kernel, make, n):
    s, d = make()
    for o in (tcamd.ORIENT_ID, tcamd.ORIENT_DEGREE):
        g = ctx.graph(s, d, n).orient(o)
        want = g.count(auto_thresholds=[64, 2048, 0, 8]).count
        other = {"bisson": {"bitmap_min_deg": 64}, "tricore": {"tricore_parts": 2}, "fox": {"fox_max_lanes": 64}}[kernel]
        for args in ({}, {"grid_size": 3}, other):
            assert g.count(kernel, **args).count == want
        g.close()
