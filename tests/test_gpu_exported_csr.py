"""A CSR whose device addresses were given out stays as it is while work on
another stream reads it: orienting the graph anew, or closing it, waits."""
import ctypes as C

import pytest

import tcamd
from graphs import rmat

pytestmark = pytest.mark.gpu

_hip = C.CDLL("libamdhip64.so.7")
_hip.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
_hip.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
_hip.hipFree.argtypes = [C.c_void_p]


@pytest.mark.parametrize("then", ["orient", "close"])
def test_reader_on_another_stream(ctx, then):
    s, d = rmat(19, 16, 8)
    with tcamd.Context(0) as reader:
        out = C.c_void_p()
        assert _hip.hipMalloc(C.byref(out), 8) == 0
        try:
            for _ in range(3):
                g = ctx.graph(s, d).orient(tcamd.ORIENT_DEGREE)
                want, n = g.count().count, g.info().n
                rp, col = C.c_void_p(), C.c_void_p()
                assert tcamd._lib.tc_graph_device_csr(g._h, C.byref(rp), C.byref(col)) == 0
                # enqueued on the reader's stream, not waited for
                assert tcamd._lib.tc_count_csr_noalloc(reader.handle, rp, col, n, 64, out) == 0
                if then == "orient":
                    g.orient(tcamd.ORIENT_ID)
                g.close()
                other = ctx.graph(d, s).orient(tcamd.ORIENT_ADIR)  # takes what was let go
                assert _hip.hipDeviceSynchronize() == 0
                got = C.c_uint64()
                assert _hip.hipMemcpy(C.byref(got), out, 8, 2) == 0
                assert got.value == want
                other.close()
        finally:
            _hip.hipFree(out)
