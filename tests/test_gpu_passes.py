"""The binned id histogram and the two-pass key compaction: degree and
A-direction orientations of inputs around the sizes where they take over and
where the bins end, against the oracle."""
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
