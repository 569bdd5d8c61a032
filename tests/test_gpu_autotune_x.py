"""The autotuner times the x lines of a substep as the substep launches them, all
three components (one of them is a third of the time, so 60% of what the per-kernel
timers give for a substep tells the two apart); and where only the interpolations
are planned in chunks (FP64 planes of 30000 lines or more), with every segment
count of the derivatives."""
import re

import numpy as np
import pytest

from opentbl_amd import config, ic
from opentbl_amd.lib import GpuBox, OTBL_MIXED

pytestmark = pytest.mark.gpu


def tuned(nx, ny, nz, **kw):
    cfg = config.small(name="tx", nx=nx, ny=ny, nz=nz, Lx=8.0 * nx / 32, kzmax=6)
    gb = GpuBox(cfg, ic.make_state(cfg), **kw)
    before = {n: gb.get(n) for n in ("u", "v", "w", "p")}
    rep = gb.autotune(5)
    print(rep, flush=True)
    for k, a in before.items():
        assert np.array_equal(gb.get(k), a), k
    return gb, {k: float(v) for k, v in re.findall(r"(\S+)=([\d.]+)ms", rep)}


@pytest.mark.parametrize("nx,nz,kw", [(500, 252, {}), (500, 256, {"precision": OTBL_MIXED})], ids=["fp64", "mixed"])
def test_three_components(nx, nz, kw):
    gb, ms = tuned(nx, 96, nz, **kw)
    gb.close()
    cfg = config.small(name="tx", nx=nx, ny=96, nz=nz, Lx=8.0 * nx / 32, kzmax=6)
    gb = GpuBox(cfg, ic.make_state(cfg), **kw)
    gb.step(2)
    gb.kprof(1)
    gb.step(3)
    rep = gb.kprof_report()
    gb.close()
    substep = sum(rep[k][1] for k in ("interpxx", "difvisxx")) / 9
    print(f"a substep's x lines {substep:.4f} ms, tuner {ms['xchunk']:.4f} ms", flush=True)
    assert ms["xchunk"] >= 0.6 * substep


def test_chunked_interpolation_with_segments():
    gb, ms = tuned(130, 40, 1120)
    nseg = sum(bool(re.fullmatch(r"xseg\d+", k)) for k in ms)
    assert nseg > 1 and "xchunk" not in ms
    assert all(f"xchunk+xseg{q + 1}" in ms for q in range(nseg)), ms
    gb.step(1)
    assert all(np.isfinite(gb.get(k)).all() for k in ("u", "v", "w", "p"))
    gb.close()
