"""x lines split over the wavefronts of a workgroup: interpxx and difvisxx
against the CPU FP64 oracle on random fields, at the line lengths where the
plan changes (the shortest lines, one span full or with one plane in its last
chunk, two and more spans), and whole RK3 steps against the windowed kernels
(OTBL_X_WINDOW) in both precisions.  Tolerances as for the other x-line kernels
(1e-12 for an operator; mixed velocities 1e-6 of the largest)."""
import numpy as np
import pytest

from opentbl_amd import config, ic
from opentbl_amd.lib import DevArray, GpuBox, OTBL_MIXED

pytestmark = pytest.mark.gpu


def rel(a, b):
    s = max(np.abs(b).max(), 1e-300)
    return float(np.abs(np.asarray(a) - np.asarray(b)).max() / s)


def box_of(nx, nz=24):
    cfg = config.small(name=f"xc{nx}", nx=nx, ny=40, nz=nz, Lx=8.0 * nx / 32)
    return cfg, ic.make_state(cfg)


@pytest.mark.parametrize("nx", [16, 32, 33, 64, 65, 129, 160, 161, 320, 321, 384, 385, 700, 1025])
def test_operators(nx, oracle_lib):
    cfg, st = box_of(nx)
    ob, gb = oracle_lib.OracleBox(cfg, st), GpuBox(cfg, st)
    assert gb.paths()["xchunk"] != "0"
    ptr = oracle_lib.ptr
    rng = np.random.default_rng(nx)
    for R, which in ((cfg.ny + 1, 1), (cfg.ny, 0), (cfg.ny + 1, 0)):
        g, q = (np.ascontiguousarray(rng.standard_normal((nx, R, cfg.nz1))) for _ in range(2))
        oi, od = np.zeros_like(g), np.zeros_like(g)
        ob.op("interpxx", ptr(g), ptr(oi), R, which)
        ob.op("difvisxx", ptr(g), ptr(q), ptr(od), R, which)
        dg, dq, d1, d2 = DevArray.from_host(g), DevArray.from_host(q), DevArray(g.size), DevArray(g.size)
        gb.op("interpxx", dg.ptr, d1.ptr, R, which)
        gb.op("difvisxx", dg.ptr, dq.ptr, d2.ptr, R, which)
        e = rel(d1.to_host().reshape(g.shape), oi), rel(d2.to_host().reshape(g.shape), od)
        assert max(e) < 1e-12, (R, which, e)
    gb.close()


@pytest.mark.parametrize("nx,mixed", [(97, False), (385, False), (130, True), (385, True), (700, True)])
def test_steps_match_windowed(nx, mixed, monkeypatch):
    cfg, st = box_of(nx)
    prec = {"precision": OTBL_MIXED} if mixed else {}
    new = GpuBox(cfg, st, graphs=True, **prec)
    monkeypatch.setenv("OTBL_X_WINDOW", "1")
    old = GpuBox(cfg, st, graphs=True, **prec)
    assert new.paths()["xchunk"] != "0" and old.paths()["xchunk"] == "0"
    new.step(2)
    old.step(2)
    f = {n: (new.get(n), old.get(n)) for n in ("u", "v", "w", "p")}
    new.close()
    old.close()
    scale = max(np.abs(f[n][1]).max() for n in "uvw")
    errs = {n: float(np.abs(f[n][0] - f[n][1]).max() / scale) for n in "uvw"}
    assert all(e < (1e-6 if mixed else 1e-12) for e in errs.values()), errs
