"""Registers that decide how many wavefronts a SIMD holds, as the compiler reports them for gfx950: a change of
the shared arithmetic that costs a kernel family a wavefront is a loss of speed that no result shows."""

import re
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "fullwave25_amd" / "csrc"


def occupancy(source: str) -> dict[str, int]:
    """Wavefronts a SIMD by kernel (mangled name)."""
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(hipcc).exists():
        pytest.skip("hipcc not found")
    cmd = [hipcc, "-O3", "--offload-arch=gfx950", "-std=c++17", "-fPIC", "-Xclang", "-target-feature", "-Xclang",
           "-packed-fp32-ops", "-Rpass-analysis=kernel-resource-usage", "--offload-device-only", "-c", "-o", "/dev/null",
           str(CSRC / source)]
    res = subprocess.run(cmd, capture_output=True, text=True, timeout=600)
    assert res.returncode == 0, res.stderr[-2000:]
    out, name = {}, None
    for line in res.stderr.splitlines():
        if m := re.search(r"Function Name: (\S+)", line):
            name = m.group(1)
        elif (m := re.search(r"Occupancy \[waves/SIMD\]: (\d+)", line)) and name:
            out[name] = int(m.group(1))
    return out


def test_marching_velocity_kernels_hold_five_wavefronts():
    """The 2D marching velocity kernels on isotropic media (4256 x 2208 cells: 103 us with five, 150 with four)."""
    occ = {k: v for k, v in occupancy("fw_kernels_stream.hip").items() if re.search(r"k_velocity_2dILi\d+ELb[01]ELb1ELb[01]E", k)}
    assert len(occ) == 12  # 64, 128, 256 lanes; one sound speed or more; maps or codes
    assert min(occ.values()) >= 5, occ
