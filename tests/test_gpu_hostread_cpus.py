"""Host threads widen a mixed box's fields only where the reading thread may use six
CPUs or more; bound to fewer, a read starts none and the GPU widens.  The same
doubles either way."""
import os

import numpy as np
import pytest

from opentbl_amd import config, ic
from opentbl_amd.lib import GpuBox, OTBL_MIXED

pytestmark = pytest.mark.gpu


def threads():
    return len(os.listdir("/proc/self/task"))


@pytest.mark.parametrize("ncpu", [1, 5, 8])
def test_threads_follow_affinity(ncpu, monkeypatch):
    mine = os.sched_getaffinity(0)
    if len(mine) < ncpu:
        pytest.skip(f"needs {ncpu} CPUs")
    cfg = config.small(name="rc", nx=130, ny=40, nz=12, Lx=8.0 * 130 / 32, kzmax=3)
    st = ic.make_state(cfg)
    ref = GpuBox(cfg, st, precision=OTBL_MIXED)
    monkeypatch.setenv("OTBL_READ_MIN", "1")
    box = GpuBox(cfg, st, precision=OTBL_MIXED)
    want = ref.get("u")
    before = threads()
    os.sched_setaffinity(0, sorted(mine)[:ncpu])
    try:
        got = box.get("u")
        started = threads() - before
    finally:
        os.sched_setaffinity(0, mine)
    ref.close()
    box.close()
    assert np.array_equal(got, want)
    assert started == 0 if ncpu < 6 else started > 0, started
    assert threads() <= before
