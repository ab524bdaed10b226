"""tc_ctx_release_memory: what a closed graph leaves with its context goes back
to the system, and the context goes on counting."""
import ctypes as C

import pytest

import oracle as orc
import tcamd

pytestmark = pytest.mark.gpu

_hip = C.CDLL("libamdhip64.so.7")


def free_bytes():
    free, total = C.c_size_t(), C.c_size_t()
    assert _hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def test_release_memory():
    s, d = tcamd.gen_er(200_000, 4_000_000, 1)
    want = orc.pipeline_count(s, d, "degree")[0]
    with tcamd.Context(0) as c:
        for _ in range(2):
            g = c.graph(s, d).orient(tcamd.ORIENT_DEGREE)
            assert g.count().count == want
            g.close()
            kept = free_bytes()
            c.release_memory()
            assert free_bytes() - kept >= 8 * len(s)  # the records, at least
