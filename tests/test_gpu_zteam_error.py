"""Error of a mixed substep's right-hand sides against an FP64 box that starts from
the same (FP32) fields: with several z rows per wavefront no larger than with the
LDS transforms (OTBL_Z_LDS).  Root mean squares over whole fields (at least 1e5
values), whose sampling error is below 1%; 10% are left for transforms of the same
length whose roundings number the same but fall elsewhere."""
import numpy as np
import pytest

from opentbl_amd import config, ic
from opentbl_amd.lib import GpuBox, OTBL_MIXED

pytestmark = pytest.mark.gpu

STATE = ("u", "v", "w", "p", "rhsupa", "rhsvpa", "rhswpa")


@pytest.mark.parametrize("nz", [54, 98, 126, 160, 224, 378, 640, 768, 980])
def test_rhs_error(nz, monkeypatch):
    cfg = config.small(name=f"ze{nz}", nx=130, ny=40, nz=nz, Lx=8.0 * 130 / 32, kzmax=min(40, nz // 3 - 1),
                       spectrum="k53")
    st = ic.make_state(cfg)
    start = GpuBox(cfg, st, precision=OTBL_MIXED)
    start.step(1)
    st = dict(st, **{n: start.get(n) for n in STATE})
    start.close()

    def rhs(**kw):
        b = GpuBox(cfg, st, **kw)
        z = int(b.paths()["zteam"])
        b.rhsp(1)
        out = {n: b.get(n) for n in STATE[4:]}
        b.close()
        return out, z

    exact, _ = rhs()
    new, zn = rhs(precision=OTBL_MIXED)
    monkeypatch.setenv("OTBL_Z_LDS", "1")
    old, zo = rhs(precision=OTBL_MIXED)
    assert zn > 0 and zo == 0
    for n in STATE[4:]:
        e, o = (float(np.sqrt((np.abs(r[n] - exact[n]) ** 2).mean())) for r in (new, old))
        print(f"nz {nz} {n}: {e / o:.2f} of the LDS kernels' error", flush=True)
        assert e <= 1.1 * o, n
