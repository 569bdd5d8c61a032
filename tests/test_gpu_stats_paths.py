"""The statistics' row-sum kernels that the shorter lengths no longer reach by
themselves: one row per engine team (FP64 rows of 2048 points, FP32 rows of 512 and
1024) and one row per workgroup on the LDS transforms (OTBL_Z_LDS).  FP64 against the
CPU FP64 oracle at the bounds of the other row lengths (1e-10 of an accumulator's
largest value, the enstrophy at FP32 rounding); mixed against the FP64 box at the
mixed bound (1e-5), dvdx0 and dwdx0, small differences of FP32 values, against the
mean shear."""
import numpy as np
import pytest

from opentbl_amd import config, ic
from opentbl_amd.lib import GpuBox, OTBL_MIXED

pytestmark = pytest.mark.gpu


def sample(b):
    b.stats_enable()
    b.statsp()
    s, e = b.stats(), b.ens()
    b.close()
    return s, e


@pytest.mark.parametrize("nz,lds", [(2048, False), (24, True), (96, True)], ids=["engine", "lds24", "lds96"])
def test_fp64_vs_oracle(nz, lds, oracle_lib, monkeypatch):
    cfg = config.small(name=f"sp{nz}", nx=24, ny=40, nz=nz)
    st = ic.make_state(cfg)
    ob = oracle_lib.OracleBox(cfg, st)
    if lds:
        monkeypatch.setenv("OTBL_Z_LDS", "1")
    gb = GpuBox(cfg, st)
    assert gb.paths()["zteam"] == "0"
    s, e = sample(gb)
    ob.statsp()
    so, eo = ob.stats(), ob.ens()
    for n in so:
        assert np.abs(s[n] - so[n]).max() <= 1e-10 * max(np.abs(so[n]).max(), 1e-300), n
    assert np.abs(e - eo).max() <= 2e-7 * np.abs(eo).max()


@pytest.mark.parametrize("nz", [512, 1024])
def test_mixed_engine_rows(nz):
    cfg = config.small(name=f"se{nz}", nx=130, ny=40, nz=nz, Lx=8.0 * 130 / 32, kzmax=8)
    st = ic.make_state(cfg)
    sd, ed = sample(GpuBox(cfg, st))
    sm, em = sample(GpuBox(cfg, st, precision=OTBL_MIXED))
    shear = np.abs(sd["dudy0"]).max()
    for n in sd:
        d = np.abs(sm[n] - sd[n]).max()
        if n in ("dvdx0", "dwdx0"):
            assert d < 1e-7 * shear, n
        else:
            assert d < 1e-5 * max(np.abs(sd[n]).max(), 1e-300), n
    assert np.abs(em - ed).max() < 1e-5 * np.abs(ed).max()
