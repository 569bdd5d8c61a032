"""interpxx with its input as its output: where a line is one span of chunks, and in
boxes of so many lines that the windowed kernel, which takes longer lines in place,
has one segment per line (400000 lines or more).  Against the same call on two
arrays: bit for bit in chunks, to 1e-12 (the bound of an operator) between the
chunked and the windowed kernel."""
import numpy as np
import pytest

from opentbl_amd import config, ic
from opentbl_amd.lib import DevArray, GpuBox

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz", [(32, 40, 24), (384, 40, 24), (385, 383, 1568)])
def test_in_place(nx, ny, nz):
    cfg = config.small(name="ip", nx=nx, ny=ny, nz=nz, Lx=8.0 * nx / 32)
    st = ic.make_state(config.small(name="ip", nx=32, ny=ny, nz=24))  # its y grid and profiles
    for n in ("u", "v", "w", "p"):
        st[n] = np.zeros((nx, ny if n in "vp" else ny + 1, cfg.mz), np.complex128)
    gb = GpuBox(cfg, st)
    assert nx <= 384 or gb.paths()["xseg"] == "1"
    P = (ny + 1) * cfg.nz1
    rng = np.random.default_rng(nx)
    g = rng.standard_normal(min(nx * P, 1 << 22))
    g = np.resize(g, nx * P)
    a, b = DevArray.from_host(g), DevArray(g.size)
    gb.op("interpxx", a.ptr, b.ptr, ny + 1, 1)
    want = b.to_host()
    gb.op("interpxx", a.ptr, a.ptr, ny + 1, 1)
    got = a.to_host()
    gb.close()
    err = np.abs(got - want).max() / np.abs(want).max()
    assert err == 0.0 if nx <= 384 else err < 1e-12, err
