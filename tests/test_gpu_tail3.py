"""The fused tail of an FP64 box's three components in one launch (boxes whose
workgroups run in one round) and in three, on both sides of the rule (3 nz1 nx / 64
workgroups of up to 256, chunks of 4 and 8 rows), against rhs_loop2, boun and
rk_final run apart (OTBL_Y_NOTAIL): the same expressions, so bit for bit."""
import numpy as np
import pytest

from opentbl_amd import config, ic
from opentbl_amd.lib import GpuBox

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz", [(16, 40, 12), (77, 63, 24), (302, 41, 24), (303, 41, 24), (33, 64, 24),
                                      (40, 127, 24), (40, 128, 24)])
def test_tail_matches_three_passes(nx, ny, nz, monkeypatch):
    cfg = config.small(name="t3", nx=nx, ny=ny, nz=nz, Lx=8.0 * nx / 32, kzmax=3)
    st = ic.make_state(cfg)
    new = GpuBox(cfg, st)
    monkeypatch.setenv("OTBL_Y_NOTAIL", "1")
    old = GpuBox(cfg, st)
    assert new.paths()["tail"] == "1" and old.paths()["tail"] == "0"
    for b in (new, old):
        b.step(2)
    for n in ("u", "v", "w", "p", "rhsupa", "rhsvpa", "rhswpa"):
        a, o = new.get(n), old.get(n)
        assert np.isfinite(a).all()
        assert np.array_equal(a, o), n
    new.close()
    old.close()
