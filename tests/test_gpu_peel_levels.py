"""Peels of very many tiny levels: one launch runs only so many of them (2,048),
and the host goes on from the frontier that it leaves, at every way a launch can
end, against the oracle."""
import numpy as np
import pytest

import oracle as orc
import tcamd
from test_gpu_parity import oracle_csr

pytestmark = pytest.mark.gpu


def path(n):
    v = np.arange(n - 1, dtype=np.uint32)
    return v, v + 1


def fuse(n, leaves):
    """A path that burns from one end to a hub of `leaves` paths of two vertices."""
    s, d = path(n)
    a = n + 2 * np.arange(leaves)
    s = np.concatenate([s, np.full(leaves, n - 1), a])
    d = np.concatenate([d, a, a + 1])
    return s.astype(np.uint32), d.astype(np.uint32)


# a level takes a vertex from either end: 2,048 of them end at 4,098 vertices
CASES = [lambda n=n: path(n) for n in (4095, 4096, 4097, 4098, 4099, 4100, 4101, 8194, 8196, 8198,
                                       20001)]
CASES += [lambda n=n: fuse(n, 9000) for n in (2047, 2048, 2049, 2050, 4200)]


@pytest.mark.parametrize("make", CASES)
def test_long_cascades(ctx, make):
    s, d = make()
    n = orc.num_nodes(s, d)
    srp, scol = orc.build_sym(s, d, n)
    for mode, o, key in (("adir", tcamd.ORIENT_ADIR, orc.adir_priority(n, srp, scol)),
                         ("kcore", tcamd.ORIENT_KCORE, orc.kcore(n, srp, scol)),
                         ("degeneracy", tcamd.ORIENT_DEGENERACY, orc.degeneracy(n, srp, scol)[0])):
        g = ctx.graph(s, d).orient(o)
        np.testing.assert_array_equal(g.vertex_key(), key.astype(np.int32))
        for got, want in zip(g.csr(), oracle_csr(s, d, mode)):
            np.testing.assert_array_equal(got, want)
        g.close()
