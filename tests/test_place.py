"""Placement of visibilities (rang-core_amd/csrc/wg_place.h) on the host: the
count and the scatter of the sort must find the same bucket also where w, u or v
lie within a rounding of a plane, cell or tile boundary, and the bucket is the
one of the unfused formula (wgridder.rs:1003-1031); the two passes of the tile
order must find the same ring."""

import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
CSRC = ROOT / "rang-core_amd" / "csrc"
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


def has_fma():
    try:
        return " fma " in Path("/proc/cpuinfo").read_text()
    except OSError:
        return False


@pytest.mark.skipif(not Path(HIPCC).exists(), reason="needs the HIP compiler")
@pytest.mark.skipif(not has_fma(), reason="needs a CPU with fused multiply-add")
def test_both_placements_agree_on_boundaries(tmp_path):
    # the device code's contraction mode, for a host that has the fused operation
    exe = tmp_path / "place_check"
    subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-O3", "-std=c++17", "-mfma", "-w",
                    "-ffp-contract=fast-honor-pragmas", f"-I{CSRC}", str(ROOT / "tests" / "place_check.cpp"),
                    str(CSRC / "wg_plan.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout
    calls, vis, differ, broken, off, edge, rings = map(int, out.split())
    assert calls == 4000 and edge > 1000  # the boundaries are reached
    assert (differ, broken, off) == (0, 0, 0), out
    assert rings == 0, out  # the tile order's two passes likewise
