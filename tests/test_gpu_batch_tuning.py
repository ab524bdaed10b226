"""The autotuner over a batch that is counted over 16-bit rows, whose time has
nothing to do with the task parameters: it still picks those that suit the
32-bit tasks of the per-graph launches."""
import pytest

import tcamd
from tcamd import batch as tbatch

pytestmark = pytest.mark.gpu


def test_tuned_tasks_suit_the_pergraph_launches(ctx):
    b = ctx.batch(tbatch.make_batch(48, 5))

    def ms(s):
        b.count_pergraph(s)
        return min(b.count_pergraph(s)[1]["ms_count"] for _ in range(3))

    times = {d: ms(dict(wave_max_deg=d)) for d in (16, 32, 64, 128, 256, 512)}
    # (7.6 ms with 32, 10 with 64, 30 with 128, 44 with 256 and 512)
    assert max(times.values()) > 3 * min(times.values())
    for _ in range(4):
        s = b.autotune()
        assert s.form == tcamd.BATCH_WORKLIST
        assert ms(s) <= 2 * min(times.values()), (s.as_dict(), times)
    b.close()
