"""Error of the chunked x interpolation (FP64) on fields near 1, as the mean flow
is, against the same factored system solved in extended precision: no larger than
the windowed kernel's (OTBL_X_WINDOW).  Root mean squares; 10% for the correction by
the neighbouring chunks' carries, one more rounding of a term below a third of the
value beside each chunk's ends (a variance of at most 1/9 of the final rounding's on
at most half of the rows)."""
import numpy as np
import pytest

from opentbl_amd import config, ic
from opentbl_amd.lib import DevArray, GpuBox

pytestmark = pytest.mark.gpu

L = np.longdouble


def interpxx(gb, g, which_u):
    """The interpolation of g (nx, lines) by the box's own coefficients."""
    nx = g.shape[0]
    a = gb.coef("inxu" if which_u else "inxv").astype(L)
    c = gb.coef("cofiux" if which_u else "cofivx").astype(L)
    b = gb.coef("inbx").astype(L)
    hi, lo = (1, 2) if which_u else (0, 3)
    g = g.astype(L)
    r = np.empty_like(g)
    r[1:-1] = c[0, 1:-1, None] * g[1:-1] + c[1, 1:-1, None] * g[2:]
    r[0] = sum(b[lo, k] * g[k] for k in range(4))
    r[-1] = sum(b[hi, k] * g[nx - 1 - k] for k in range(4))
    for i in range(1, nx):
        r[i] += a[0, i] * r[i - 1]
    r[-1] *= a[1, -1]
    for i in range(nx - 2, -1, -1):
        r[i] = (r[i] - a[2, i] * r[i + 1]) * a[1, i]
    return r


@pytest.mark.parametrize("nx", [32, 64, 96, 161, 384, 385, 700])
def test_interpolation_error(nx, monkeypatch):
    cfg = config.small(name=f"xe{nx}", nx=nx, ny=40, nz=24, Lx=8.0 * nx / 32)
    st = ic.make_state(cfg)
    new = GpuBox(cfg, st)
    monkeypatch.setenv("OTBL_X_WINDOW", "1")
    old = GpuBox(cfg, st)
    assert new.paths()["xchunk"] != "0" and old.paths()["xchunk"] == "0"
    rng = np.random.default_rng(nx)
    x = np.linspace(0.0, 1.0, nx)[:, None, None]
    for R, which in ((cfg.ny + 1, 1), (cfg.ny, 0)):
        k = rng.integers(1, max(2, nx // 16), (1, R, cfg.nz1))
        g = np.ascontiguousarray(1.0 + 0.05 * np.sin(2 * np.pi * (k * x + rng.uniform(0, 1, (1, R, cfg.nz1)))))
        want = interpxx(new, g.reshape(nx, -1), which)
        dg, err = DevArray.from_host(g), []
        for b in (new, old):
            d = DevArray(g.size)
            b.op("interpxx", dg.ptr, d.ptr, R, which)
            err.append(float(np.sqrt(((d.to_host().reshape(nx, -1) - want) ** 2).mean())))
        print(f"nx {nx} which {which}: {err[0]:.2e} / {err[1]:.2e} = {err[0] / err[1]:.3f}", flush=True)
        assert err[0] <= 1.1 * err[1], (which, err)
    new.close()
    old.close()
