"""The mean-flow mode of the pressure solve in the launch of the other modes
(y chunks of up to 8 rows: ny - 1 <= 256) and in one of its own (longer chunks),
and the implicit factors in the launch of the inflow statistics, against the
marched columns (OTBL_Y_MARCH: every mode in one marching launch), at the sizes on
both sides of the rule and with more mean-flow columns than one workgroup holds.
FP64, one step: 1e-10 of a field's largest value, the bound of a step against the
oracle."""
import numpy as np
import pytest

from opentbl_amd import config, ic
from opentbl_amd.lib import GpuBox

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz", [(16, 40, 12), (130, 41, 12), (40, 257, 24), (40, 258, 24), (300, 65, 16)])
def test_step_matches_marching(nx, ny, nz, monkeypatch):
    cfg = config.small(name="pm", nx=nx, ny=ny, nz=nz, Lx=8.0 * nx / 32, kzmax=3)
    st = ic.make_state(cfg)
    new = GpuBox(cfg, st)
    monkeypatch.setenv("OTBL_Y_MARCH", "1")
    old = GpuBox(cfg, st)
    for b in (new, old):
        b.step(1)
    for n in ("u", "v", "w", "p"):
        a, o = new.get(n), old.get(n)
        assert np.isfinite(a).all()
        assert np.abs(a - o).max() <= 1e-10 * np.abs(o).max(), n
    new.close()
    old.close()
