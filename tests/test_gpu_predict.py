"""The pressure-gradient predictor formed inside the final y update (chunked
solver) against the pass of its own that the marched columns keep
(OTBL_Y_MARCH), at the edges of its chunks: the last row, or the last but one,
of a column at the start of a chunk, the shortest and a longer chunk, the
three-pass tail, and on FP32 half-wave chunks several mean-flow columns per
workgroup.

FP64: two steps agree to 1e-10 of a field's largest value, the bound of a step
against the oracle.  Mixed: 1e-6 of the largest velocity, its bound against
FP64."""
import numpy as np
import pytest

from opentbl_amd import config, ic
from opentbl_amd.lib import GpuBox, OTBL_MIXED

pytestmark = pytest.mark.gpu


def box(nx, ny, nz):
    cfg = config.small(name="pred", nx=nx, ny=ny, nz=nz, Lx=8.0 * nx / 32, kzmax=min(4, nz // 3 - 1))
    return cfg, ic.make_state(cfg)


def fields(b):
    out = {n: b.get(n) for n in ("u", "v", "w", "p", "rhsupa", "rhsvpa", "rhswpa")}
    b.close()
    assert all(np.isfinite(a).all() for a in out.values())
    return out


@pytest.mark.parametrize("nx,ny,nz", [(16, 44, 12), (21, 45, 24), (33, 63, 24), (20, 128, 24), (16, 129, 64)])
@pytest.mark.parametrize("tail", [True, False], ids=["tail", "apart"])
def test_predictor_fp64(nx, ny, nz, tail, monkeypatch):
    cfg, st = box(nx, ny, nz)
    if not tail:
        monkeypatch.setenv("OTBL_Y_NOTAIL", "1")
    new = GpuBox(cfg, st)
    assert new.paths()["y"].startswith("chunk")
    monkeypatch.setenv("OTBL_Y_MARCH", "1")
    old = GpuBox(cfg, st)
    assert old.paths()["y"].startswith("march")
    for b in (new, old):
        b.step(2)
    a, o = fields(new), fields(old)
    for n in a:
        assert np.abs(a[n] - o[n]).max() <= 1e-10 * np.abs(o[n]).max(), n


@pytest.mark.parametrize("nx,ny,nz,half", [(130, 44, 12, True), (130, 45, 16, True), (150, 97, 64, True),
                                           (130, 129, 24, True), (130, 45, 12, False)])
def test_predictor_mixed(nx, ny, nz, half, monkeypatch):
    cfg, st = box(nx, ny, nz)
    if not half:
        monkeypatch.setenv("OTBL_Y_HALF", "0")
    new, old = GpuBox(cfg, st, precision=OTBL_MIXED), GpuBox(cfg, st)
    assert new.paths()["y"].endswith("h") == half
    for b in (new, old):
        b.step(2)
    a, o = fields(new), fields(old)
    scale = max(np.abs(o[n]).max() for n in ("u", "v", "w"))
    for n in ("u", "v", "w"):
        assert np.abs(a[n] - o[n]).max() <= 1e-6 * scale, n
