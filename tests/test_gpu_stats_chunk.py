"""The statistics' x and y lines split over the wavefronts of a workgroup and
their row sums with several rows per wavefront, against the kernels with one
thread per line (OTBL_STATS_MARCH) and one row per workgroup (OTBL_Z_LDS), at the
lengths where the plans change: one span and more of x lines, the shortest and
longest y chunks, a last y chunk of one row, two- and three-pass rows.

FP64: the sums of a sample agree to 1e-10 of the accumulator's largest value
(second derivatives of a field amplify its round-off by up to 1e4 on these
grids).  Mixed: both keep FP32 intermediate fields, whose rounding differs
where the kernels' FP64 results differ by their last bit; 1e-4 of the largest
value."""
import numpy as np
import pytest

from opentbl_amd import config, ic
from opentbl_amd.lib import GpuBox, OTBL_MIXED

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz,mixed", [(16, 40, 12, False), (33, 49, 64, False), (130, 40, 98, False),
                                            (385, 41, 24, False), (700, 40, 24, False), (40, 383, 24, False),
                                            (130, 97, 160, True), (400, 40, 54, True)])
def test_sample_matches_marching(nx, ny, nz, mixed, monkeypatch):
    cfg = config.small(name="sc", nx=nx, ny=ny, nz=nz, Lx=8.0 * nx / 32, kzmax=min(4, nz // 3 - 1))
    st = ic.make_state(cfg)
    prec = {"precision": OTBL_MIXED} if mixed else {}
    new = GpuBox(cfg, st, **prec)
    new.step(1)
    state = {n: new.get(n) for n in ("u", "v", "w", "p")}
    new.stats_enable()
    monkeypatch.setenv("OTBL_STATS_MARCH", "1")
    monkeypatch.setenv("OTBL_Z_LDS", "1")
    old = GpuBox(cfg, dict(st, **state), **prec)
    old.stats_enable()
    for b in (new, old):
        b.statsp()
    a, o = new.stats(), old.stats()
    ea, eo = new.ens(), old.ens()
    new.close()
    old.close()
    tol = 1e-4 if mixed else 1e-10
    errs = {n: float(np.abs(a[n] - o[n]).max() / max(np.abs(o[n]).max(), 1e-300)) for n in a}
    worst = max(errs, key=errs.get)
    assert errs[worst] < tol, (worst, errs[worst])
    assert float(np.abs(ea - eo).max() / np.abs(eo).max()) < (1e-4 if mixed else 1e-6)
