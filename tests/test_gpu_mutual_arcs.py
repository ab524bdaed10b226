"""k-cliques of a stage file whose CSR holds both arcs of an edge.  The loader
accepts one (rows ascending, loop-free, in range), and every path over bit
matrices counts, over all roots u, the (k-1)-cliques of the edges inside N+(u),
an edge with both arcs being one edge."""
import struct
from itertools import combinations
from math import comb

import numpy as np
import pytest

import tcamd

pytestmark = pytest.mark.gpu


def load(ctx, tmp_path, rows):
    rp = np.cumsum([0] + [len(r) for r in rows]).astype(np.uint32)
    col = np.concatenate([np.sort(r) for r in rows]).astype(np.uint32)
    p = tmp_path / "mutual.csr"
    p.write_bytes(struct.pack("<8sIIQiI", b"TCAMDCSR", 1, len(rows), len(col), tcamd.ORIENT_ID, 0)
                  + rp.tobytes() + col.tobytes())
    return ctx.load_csr(str(p))


# one-word rows at and beyond half their edge list (46: 2 * 990 arcs of 2,016), full
# rows of one word, and every wider form
@pytest.mark.parametrize("d", [3, 45, 46, 63, 64, 65, 128, 129, 257, 513])
def test_root_over_mutual_clique(ctx, tmp_path, d):
    inner = np.arange(1, d + 1)
    g = load(ctx, tmp_path, [inner] + [inner[inner != v] for v in inner])
    for k in (4, 5):
        want = comb(d, k - 1) + d * comb(d - 1, k - 1)
        assert g.kclique(k, tcamd.KCL_PIVOT).count == want
        assert g.kclique(k).count == want
        assert g.kclique_roots(k, np.arange(d + 1, dtype=np.uint32)).count == want
    assert g.kclique_roots(3, np.arange(d + 1, dtype=np.uint32)).count == \
        comb(d, 2) + d * comb(d - 1, 2)
    g.close()


def brute(rows, k):
    sets = [set(r.tolist()) for r in rows]
    total = 0
    for r in rows:
        def grow(cand, left):
            if left == 0:
                return 1
            return sum(grow([y for y in cand[i + 1:] if y in sets[x] or x in sets[y]], left - 1)
                       for i, x in enumerate(cand))
        total += grow(sorted(r.tolist()), k - 1)
    return total


@pytest.mark.parametrize("n,both", [(24, 0.2), (60, 0.5), (90, 0.05)])
def test_some_mutual_arcs(ctx, tmp_path, n, both):
    rng = np.random.default_rng(n)
    rows = [[] for _ in range(n)]
    for a, b in combinations(range(n), 2):
        x = rng.random()
        if x < 0.35 + both / 2:
            rows[a].append(b)
        if x > 0.35 - both / 2 and x < 0.7:
            rows[b].append(a)
    rows = [np.array(r, np.int64) for r in rows]
    assert any(a in rows[b] for a in range(n) for b in rows[a])
    g = load(ctx, tmp_path, rows)
    for k in (4, 5):
        want = brute(rows, k)
        assert g.kclique(k).count == want
        assert g.kclique(k, tcamd.KCL_PIVOT).count == want
        assert g.kclique_roots(k, np.arange(n, dtype=np.uint32)).count == want
    g.close()
