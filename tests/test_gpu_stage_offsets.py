"""Stage files whose row offsets rise beyond the arcs before they fall back: the
loader refuses them without reading past the arcs."""
import struct

import numpy as np
import pytest

import tcamd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rp", [[0, 1 << 30, 2, 2], [0, 3, 2, 2], [0, 2, 0xFFFFFFFF, 2], [0, 2, 1, 2]])
def test_offsets_beyond_the_arcs(ctx, tmp_path, rp):
    p = tmp_path / "bad.csr"
    p.write_bytes(struct.pack("<8sIIQiI", b"TCAMDCSR", 1, 3, 2, tcamd.ORIENT_ID, 0)
                  + np.array(rp, np.uint32).tobytes() + np.array([1, 2], np.uint32).tobytes())
    with pytest.raises(tcamd.TCError) as e:
        ctx.load_csr(str(p))
    assert e.value.status == tcamd.ERR_FORMAT
