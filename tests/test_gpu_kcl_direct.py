"""The direct k-clique path (k <= 5, roots of up to 512 out-neighbours): every
width of the bit matrix and its borders, near-complete roots, and several
workgroups per root, against closed forms, the oracle and the pivot path."""
from math import comb

import numpy as np
import pytest

import oracle as orc
import tcamd
from graphs import rmat

pytestmark = pytest.mark.gpu


def complete(n):
    u, v = np.triu_indices(n, 1)
    return u.astype(np.uint32), v.astype(np.uint32)


@pytest.mark.parametrize("n", [3, 4, 5, 33, 64, 65, 66, 129, 130, 192, 194, 257, 258, 322, 385, 449,
                               512, 513, 514])
def test_complete_graphs(ctx, n):
    g = ctx.graph(*complete(n)).orient(tcamd.ORIENT_ID)
    for k in (4, 5):
        assert g.kclique(k).count == comb(n, k)
        assert g.kclique_roots(k, np.arange(n, dtype=np.uint32)).count == comb(n, k)
    assert g.kclique_roots(3, np.arange(n, dtype=np.uint32)).count == comb(n, 3)
    g.close()


@pytest.mark.parametrize("n,keep", [(40, 0.9), (120, 0.7), (120, 0.995), (200, 0.5), (250, 0.998),
                                    (330, 0.4), (400, 0.999), (510, 0.3)])
def test_dense_graphs_match_pivot(ctx, n, keep):
    s, d = complete(n)
    m = np.random.default_rng(n).random(len(s)) < keep
    p = np.random.default_rng(n + 1).permutation(n).astype(np.uint32)
    g = ctx.graph(p[s[m]], p[d[m]], n)
    for o in (tcamd.ORIENT_ID, tcamd.ORIENT_DEGENERACY):
        g.orient(o)
        for k in (4, 5):
            want = g.kclique(k, tcamd.KCL_PIVOT).count
            assert g.kclique(k).count == want
            assert g.kclique_roots(k, np.arange(n, dtype=np.uint32)).count == want
    g.close()


@pytest.mark.parametrize("scale,ef", [(9, 8), (12, 16), (13, 40)])
@pytest.mark.parametrize("k", [4, 5])
def test_skewed(ctx, scale, ef, k):
    s, d = rmat(scale, ef, scale)
    for o in (tcamd.ORIENT_DEGENERACY, tcamd.ORIENT_DEGREE):
        g = ctx.graph(s, d, 1 << scale).orient(o)
        want = g.kclique(k, tcamd.KCL_MERGE).count
        assert g.kclique(k).count == want
        assert g.kclique(k).count == want  # over the kept order
        g.close()
    if scale == 9:
        _, rp, col = orc.pipeline_count(s, d, "degree")
        assert want == orc.kclique(rp, col, k)


def test_order_follows_the_graph(ctx):
    # the kept order of the roots is rebuilt when the orientation changes
    s, d = rmat(11, 24, 4)
    g = ctx.graph(s, d, 1 << 11)
    counts = set()
    for o in (tcamd.ORIENT_DEGREE, tcamd.ORIENT_ID, tcamd.ORIENT_DEGENERACY, tcamd.ORIENT_ID):
        counts.add(g.orient(o).kclique(5).count)
    assert len(counts) == 1
    g.close()
