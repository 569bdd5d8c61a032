"""z transforms with several rows per wavefront (even row lengths 12 to 1024
of factors 2, 3, 5, 7): fourxz against the CPU FP64 oracle's c2r / r2c, and
whole RK3 steps against the LDS kernels (OTBL_Z_LDS) in both precisions.
Lengths: the shortest and the longest, two and three passes, rows that leave
lanes of a wavefront idle or its last butterflies partly filled, and those
that hold most values per lane.

Tolerances: FP64 as the other z transforms (1e-12 of an operator's largest
value, 1e-10 after a step); mixed: velocities within 1e-6 of the largest, the
bound that the mixed substep is held to against FP64."""
import numpy as np
import pytest

from opentbl_amd import config, ic
from opentbl_amd.lib import DevArray, GpuBox, OTBL_MIXED

pytestmark = pytest.mark.gpu


def rel(a, b):
    s = max(np.abs(b).max(), 1e-300)
    return float(np.abs(np.asarray(a) - np.asarray(b)).max() / s)


def box_of(nz, nx=16, **kw):
    cfg = config.small(name=f"zt{nz}", nx=nx, ny=41, nz=nz, Lx=8.0 * nx / 32, kzmax=min(40, nz // 3 - 1))
    return cfg, ic.make_state(cfg)


@pytest.mark.parametrize("nz", [12, 14, 24, 54, 64, 98, 126, 160, 224, 250, 378, 640, 648, 768, 980, 1008])
@pytest.mark.parametrize("nrows", [1, 37])
def test_fourxz(nz, nrows, oracle_lib):
    cfg, st = box_of(nz)
    ob = oracle_lib.OracleBox(cfg, st)
    gb = GpuBox(cfg, st)
    assert int(gb.paths()["zteam"]) > 0
    rng = np.random.default_rng(nz)
    L, ptr = oracle_lib.lib(), oracle_lib.ptr
    fou, phys = rng.standard_normal((nrows, cfg.nz1)), rng.standard_normal((nrows, nz))
    phys_o, fou_o = np.zeros((nrows, nz)), np.zeros((nrows, cfg.nz1))
    for r in range(nrows):
        L.oc_c2r(ob.h, ptr(np.ascontiguousarray(fou[r])), ptr(phys_o[r]))
        L.oc_r2c(ob.h, ptr(np.ascontiguousarray(phys[r])), ptr(fou_o[r]))
    dfou, dphys = DevArray.from_host(fou), DevArray(nrows * nz)
    gb.op("fourxz", dfou.ptr, dphys.ptr, 1, nrows)
    e1 = rel(dphys.to_host().reshape(nrows, nz), phys_o)
    dphys2, dfou2 = DevArray.from_host(phys), DevArray(nrows * cfg.nz1)
    gb.op("fourxz", dfou2.ptr, dphys2.ptr, -1, nrows)
    e2 = rel(dfou2.to_host().reshape(nrows, cfg.nz1), fou_o)
    gb.close()
    assert e1 < 1e-12 and e2 < 1e-12, (e1, e2)


@pytest.mark.parametrize("mixed", [False, True], ids=["fp64", "mixed"])
@pytest.mark.parametrize("nz", [12, 54, 98, 160, 250, 378, 648, 980])
def test_steps_match_lds_kernels(nz, mixed, monkeypatch):
    cfg, st = box_of(nz, nx=130)
    prec = {"precision": OTBL_MIXED} if mixed else {}
    new = GpuBox(cfg, st, **prec)
    monkeypatch.setenv("OTBL_Z_LDS", "1")
    old = GpuBox(cfg, st, **prec)
    assert int(new.paths()["zteam"]) > 0 and old.paths()["zteam"] == "0"
    new.step(2)
    old.step(2)
    f = {n: (new.get(n), old.get(n)) for n in ("u", "v", "w", "p")}
    t, to = new.time(), old.time()
    new.close()
    old.close()
    if mixed:
        scale = max(np.abs(f[n][1]).max() for n in "uvw")
        errs = {n: float(np.abs(f[n][0] - f[n][1]).max() / scale) for n in "uvw"}
        assert all(e < 1e-6 for e in errs.values()), errs
        assert abs(t[1] - to[1]) <= 1e-5 * to[1]
    else:
        errs = {n: rel(*f[n]) for n in f}
        assert all(errs[n] < 1e-10 for n in "uvw") and errs["p"] < 1e-8, errs
        assert abs(t[1] - to[1]) <= 1e-12 * to[1]
