"""The binned id histogram, the two-pass key compaction and the peel's small
levels: orientations of inputs around the sizes where they take over and where
the bins end, against the oracle."""
import numpy as np
import pytest

import oracle as orc
import tcamd
from graphs import rmat
from test_gpu_parity import oracle_csr

pytestmark = pytest.mark.gpu


def check(ctx, s, d, mode, orient):
    g = ctx.graph(s, d).orient(orient)
    rp, col = g.csr()
    rp_o, col_o = oracle_csr(s, d, mode)
    np.testing.assert_array_equal(rp, rp_o)
    np.testing.assert_array_equal(col, col_o)
    g.close()


# records: 2^19 is where 2 m ids are binned, 2^20 where m keys are compacted; ids:
# one bin, the first of the next, 256 bins, beyond
@pytest.mark.parametrize("n", [16384, 16385, 65537, 1 << 22, (1 << 22) + 1])
@pytest.mark.parametrize("m", [(1 << 19) - 1, 1 << 19, (1 << 20) + 8191])
def test_degree_orientation(ctx, n, m):
    s, d = tcamd.gen_er(n, m - 1, 3)
    s, d = np.append(s, np.uint32(n - 1)), np.append(d, np.uint32(0))  # the last id occurs
    dup = np.random.default_rng(n).integers(0, m, m // 16)             # duplicates to drop
    s[dup], d[dup] = s[dup[::-1]], d[dup[::-1]]
    check(ctx, s, d, "degree", tcamd.ORIENT_DEGREE)


def test_skewed(ctx):
    s, d = rmat(17, 16, 5)
    check(ctx, s, d, "degree", tcamd.ORIENT_DEGREE)
    check(ctx, s, d, "adir", tcamd.ORIENT_ADIR)


def path(n):
    v = np.arange(n - 1, dtype=np.uint32)
    return v, v + 1


def star(leaves, hubs=1):
    """Leaves on hubs that form a clique: one level takes all leaves."""
    u, v = np.triu_indices(hubs + 4, 1)
    leaf = np.arange(leaves) + hubs + 4
    return (np.concatenate([u, leaf]).astype(np.uint32),
            np.concatenate([v, np.arange(leaves) % hubs]).astype(np.uint32))


def ring_of(n, reach):
    """Every vertex joined to the next `reach`: whole levels of one row length."""
    u = np.repeat(np.arange(n), reach)
    return u.astype(np.uint32), ((u + np.tile(np.arange(1, reach + 1), n)) % n).astype(np.uint32)


@pytest.mark.parametrize("make", [lambda: path(2), lambda: path(5001), lambda: star(1023), lambda: star(1024),
                                  lambda: star(1025), lambda: star(3000, 40), lambda: star(20000, 3),
                                  lambda: ring_of(1024, 4), lambda: ring_of(1023, 5), lambda: rmat(10, 12, 3)])
def test_small_levels(ctx, make):
    s, d = make()
    for mode, o in (("adir", tcamd.ORIENT_ADIR), ("kcore", tcamd.ORIENT_KCORE)):
        check(ctx, s, d, mode, o)


@pytest.mark.parametrize("n,m", [(300_000, (1 << 20) - 1), (300_000, 1 << 20), (1_500_000, 1 << 20)])
def test_pruned(ctx, n, m):
    # keys over fewer rows than ids, packed from 2^20 records on
    s, d = tcamd.gen_er(n, m, 11)
    g = ctx.graph(s, d).orient(tcamd.ORIENT_DEGREE)
    want = g.count().count
    g.orient(tcamd.ORIENT_DEGREE, prune_deg1=True)
    assert g.info().n < n
    assert g.count().count == want
    g.close()


@pytest.mark.parametrize("m", [1, 63, 1023, 1024, 1025, 4097, 300_001, 2_100_003])
def test_largest_id(ctx, m):
    rng = np.random.default_rng(m)
    for where, side in ((0, 0), (m - 1, 0), (m // 2, 1), (m - 1, 1)):
        ends = [rng.integers(0, 5000, m).astype(np.uint32) for _ in range(2)]
        ends[side][where] = 7654
        g = ctx.graph(*ends)
        assert g.info().n == 7655
        g.close()
