"""The one-launch fused tail is for boxes whose workgroups run in one round of this
device's compute units: launches per substep, by the per-kernel timers, on both
sides of the rule."""
import ctypes

import pytest

from opentbl_amd import config, ic
from opentbl_amd.lib import GpuBox, lib

pytestmark = pytest.mark.gpu

MULTIPROCESSOR_COUNT = 63  # hipDeviceAttributeMultiprocessorCount


def compute_units():
    lib()  # its HIP runtime, not another one
    n = ctypes.c_int()
    assert ctypes.CDLL("libamdhip64.so.7").hipDeviceGetAttribute(ctypes.byref(n), MULTIPROCESSOR_COUNT, 0) == 0
    return n.value


@pytest.mark.parametrize("more", [0, 1])
def test_one_round(more):
    cus = compute_units()
    nx = cus // 3 * 64 // 16 + more  # 16 columns a plane, 64 a workgroup
    cfg = config.small(name="tc", nx=nx, ny=41, nz=24, Lx=8.0 * nx / 32)
    assert cfg.nz1 == 16
    gb = GpuBox(cfg, ic.make_state(cfg))
    gb.kprof(1)
    gb.step(1)
    n = gb.kprof_report()["rk_tail"][0]
    gb.close()
    wg = 3 * ((16 * nx + 63) // 64)
    assert (wg <= cus) == (not more)
    assert n == 3 * (3 if more else 1), (n, wg, cus)
