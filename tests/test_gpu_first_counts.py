"""Hu's and Fox's methods and per-vertex counts over the first counts of a
graph, which read the CSR, and the later ones, which stream list rows: the same
values throughout, also when other counts build the rows in between and when
the graph is oriented anew."""
import numpy as np
import pytest

import oracle as orc
import tcamd
from graphs import CASES, hub, rmat

pytestmark = pytest.mark.gpu

MAKE = {name: (make, 0) for name, make in CASES.items()}
MAKE["two parts"] = (lambda: tcamd.gen_er(72_001, 400_003, 5), 0)
MAKE["32-bit rows"] = (lambda: tcamd.gen_er(300_001, 900_001, 5), 0)
MAKE["64 vertices a block"] = (lambda: rmat(16, 8, 9), 1 << 16)
ROUNDS = 6  # three over the CSR, the one that builds the rows, and two more


@pytest.mark.parametrize("name", list(MAKE))
def test_repeated(ctx, name):
    make, n = MAKE[name]
    s, d = make()
    g = ctx.graph(s, d, n)
    for o in (tcamd.ORIENT_ID, tcamd.ORIENT_DEGREE):
        g.orient(o)
        tri = orc.count_per_vertex(*g.csr())
        for i in range(ROUNDS):
            assert g.count("hu", grid_size=(0, 1000)[i % 2]).count == tri.sum()
            assert g.count("fox").count == tri.sum()
            np.testing.assert_array_equal(g.count_per_vertex(), tri)
    g.close()


@pytest.mark.parametrize("first", ["hu", "fox", "auto", "vertex"])
def test_rows_of_another_count(ctx, first):
    s, d = MAKE["two parts"][0]()
    g = ctx.graph(s, d).orient(tcamd.ORIENT_ADIR)
    tri = orc.count_per_vertex(*g.csr())
    ops = {k: (lambda k=k: g.count(k).count) for k in ("hu", "fox", "auto", "bisson", "tricore")}
    ops["vertex"] = lambda: int(g.count_per_vertex().sum())
    for _ in range(ROUNDS):
        assert ops[first]() == tri.sum()
    for k in ops:
        assert ops[k]() == tri.sum()
    np.testing.assert_array_equal(g.count_per_vertex(), tri)
    g.close()


def test_rows_wider_than_a_slice(ctx):
    # rows of more than 2,048 entries, and blocks of one vertex and of all of them
    s, d = hub(9000, 30000)
    g = ctx.graph(s, d).orient(tcamd.ORIENT_ID)
    want = orc.count(*g.csr())
    assert g.info().max_out_degree == 9000
    for blocks in (1, 7, 9001):
        g.orient(tcamd.ORIENT_ID)  # its first count again
        assert g.count("hu", grid_size=blocks).count == want
    g.close()
