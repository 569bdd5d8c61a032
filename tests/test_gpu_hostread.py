"""Fields of a mixed box widened by the host's threads (the default for large
fields, forced here by OTBL_READ_MIN) against the GPU's widening: the same
doubles, bit for bit, for fields within one staging slot, over several slots and
over reused ones, for a host array that is not 16-byte aligned, and for two boxes
read from two threads."""
import ctypes
import threading

import numpy as np
import pytest

from opentbl_amd import config, ic
from opentbl_amd.lib import FIELDS, GpuBox, OTBL_MIXED, check, lib

pytestmark = pytest.mark.gpu

NAMES = ("u", "v", "w", "p", "rhsupa")


def boxes(nx, ny, nz, monkeypatch, n=1):
    cfg = config.small(name="read", nx=nx, ny=ny, nz=nz, Lx=8.0 * nx / 32, kzmax=3)
    st = ic.make_state(cfg)
    ref = GpuBox(cfg, st, precision=OTBL_MIXED)
    monkeypatch.setenv("OTBL_READ_MIN", "1")
    out = [GpuBox(cfg, st, precision=OTBL_MIXED) for _ in range(n)]
    for b in [ref] + out:
        b.step(1)
    return [ref] + out


@pytest.mark.parametrize("nx,ny,nz", [(130, 40, 12), (131, 97, 256), (257, 97, 512)])
def test_read_matches(nx, ny, nz, monkeypatch):
    ref, new = boxes(nx, ny, nz, monkeypatch)
    for name in NAMES:
        a, b = ref.get(name), new.get(name)
        assert np.array_equal(a, b), name
        n = lib().otbl_field_len(new.h, FIELDS[name])
        raw = np.empty(n + 3)
        at = raw[1 if raw.ctypes.data % 16 == 0 else 2:][:n]
        assert at.ctypes.data % 16 == 8
        raw[:] = 7.0
        check(lib().otbl_get_field(new.h, FIELDS[name], at.ctypes.data_as(ctypes.POINTER(ctypes.c_double))), "get")
        assert np.array_equal(at, a.view(np.float64).ravel()), name
        assert (raw == 7.0).sum() >= 3
    ref.close()
    new.close()


def test_two_threads(monkeypatch):
    ref, *two = boxes(130, 97, 512, monkeypatch, 2)
    want = ref.get("u")
    bad = []

    def read(b):
        for _ in range(5):
            if not np.array_equal(b.get("u"), want):
                bad.append(b)

    th = [threading.Thread(target=read, args=(b,)) for b in two]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad
    for b in [ref] + two:
        b.close()
