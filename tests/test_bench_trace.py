"""bench.py's kernel records against the sources (no GPU): every HIP function of a
timed kernel is known to the look-up of profiled traffic, the bytes quoted beside a
launch's time are those of all the components that it holds, and the committed
profiles list kernels that the sources have."""
import glob
import os
import re
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
import bench  # noqa: E402
from opentbl_amd import config  # noqa: E402


def hip_functions():
    out = set()
    for path in glob.glob(os.path.join(ROOT, "opentbl_amd", "csrc", "*")):
        if path.endswith((".hip", ".h")):
            out |= set(re.findall(r"__global__\s+void\s+(?:__launch_bounds__\((?:[^()]|\([^()]*\))*\)\s*)?(\w+)\(",
                                  open(path).read()))
    return out


def test_trace_names_cover_the_kernels():
    fns = hip_functions()
    assert len(fns) > 60 and "rk_tail_y" in fns
    for kname in ("products1", "products2", "interpxx", "difvisxx", "rk_final", "rk_tail", "interpyy", "rhs_loop2"):
        have = {f for f in fns if re.fullmatch(kname + r"3?_(t|z|zp|c|w|y|yh)", f)}
        names = bench.TRACE_NAMES[kname]
        names = {names} if isinstance(names, str) else set(names)
        assert have == names, (kname, have ^ names)


@pytest.mark.parametrize("kname", ["interpxx", "difvisxx"])
def test_bytes_of_a_shared_launch(kname):
    """Three components in one launch: three times the model's bytes of one."""
    m = bench.kernel_model(config.CONFIGS["zpg1536x315x1024"], 4)
    rows = bench.report("test", {"products1": (3, 1.0), kname: (3, 9.0)}, m)
    r = bench.roofline(rows, m, "none", "mixed", hbm_only=True)
    assert r["kernel"] == kname
    assert r["algorithmic_bytes"] == pytest.approx(3 * m[kname][0])
    assert r["achieved"] == pytest.approx(r["algorithmic_bytes"] / (r["avg_ms"] * 1e-3) / 1e9)


@pytest.mark.parametrize("path", sorted(glob.glob(os.path.join(ROOT, "profiles", "*.md"))), ids=os.path.basename)
def test_profiles_list_present_kernels(path):
    fns = hip_functions()
    text = open(path).read().split("## Replaced since")[0]
    names = {m.group(1) for m in re.finditer(r"^\| (\w+)(?:<[^|]*>)? \|", text, re.M)} - {"kernel"}
    names = {n for n in names if not n.startswith("__amd_rocclr")}
    assert len(names) > 3 and names <= fns, names - fns
