"""Row sums of a mixed box's statistics with several rows per wavefront against
the kernel with one row per workgroup (OTBL_Z_LDS): both take the same FP32 x and
y lines and the same FP64 mean flow through FP64 transforms, so a sample's sums
agree to FP64 round-off (1e-12 of an accumulator's largest value: a few thousand
roundings of 1e-16) and the FP32 enstrophy to its last bit (2^-23 of the largest).
Lengths: the shortest and the longest, two and three passes, lanes left idle."""
import numpy as np
import pytest

from opentbl_amd import config, ic
from opentbl_amd.lib import GpuBox, OTBL_MIXED

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nz", [12, 64, 98, 160, 250, 648, 980])
def test_mixed_row_sums(nz, monkeypatch):
    cfg = config.small(name=f"sr{nz}", nx=130, ny=40, nz=nz, Lx=8.0 * 130 / 32, kzmax=min(40, nz // 3 - 1))
    st = ic.make_state(cfg)
    new = GpuBox(cfg, st, precision=OTBL_MIXED)
    monkeypatch.setenv("OTBL_Z_LDS", "1")
    old = GpuBox(cfg, st, precision=OTBL_MIXED)
    assert int(new.paths()["zteam"]) > 0 and old.paths()["zteam"] == "0"
    for b in (new, old):
        b.stats_enable()
        b.statsp()
    a, o, ea, eo = new.stats(), old.stats(), new.ens(), old.ens()
    new.close()
    old.close()
    errs = {n: float(np.abs(a[n] - o[n]).max() / max(np.abs(o[n]).max(), 1e-300)) for n in a}
    worst = max(errs, key=errs.get)
    e = float(np.abs(ea - eo).max() / np.abs(eo).max())
    print(f"nz {nz}: {worst} {errs[worst]:.2e}, enstrophy {e:.2e}", flush=True)
    assert errs[worst] < 1e-12 and e <= 2.0 ** -23, (worst, errs[worst], e)
