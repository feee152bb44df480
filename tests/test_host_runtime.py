"""The engine's host code on a stand-in HIP runtime (tests/host_runtime.h) under AddressSanitizer, without
a GPU: what handles, graphs, point tables and adjoints free and when, and which kernels a handle launches.
tests/host_runtime_check.cpp holds the checks; a finding of the sanitizer ends the program."""

import os
import shutil
import subprocess
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
BUILD = ROOT / "tests" / "_build" / "host_runtime"
CSRC = ROOT / "fullwave25_amd" / "csrc"


@pytest.fixture(scope="module")
def driver():
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(hipcc).exists():
        pytest.skip("hipcc not found")
    exe = BUILD / "host_runtime_check"
    check = ROOT / "tests" / "host_runtime_check.cpp"
    sources = sorted(CSRC.glob("*.cpp")) + sorted(CSRC.glob("*.hip")) + [check]
    headers = [ROOT / "tests" / "host_runtime.h", ROOT / "include" / "fullwave_hip.h", *CSRC.glob("*.h")]
    newest = max(p.stat().st_mtime for p in sources + headers)
    if exe.exists() and exe.stat().st_mtime > newest:
        return exe
    BUILD.mkdir(parents=True, exist_ok=True)
    flags = ["-std=c++17", "-O1", "-g", "--offload-host-only", "-Xarch_host", "-fsanitize=address",
             "-fno-omit-frame-pointer"]

    def one(src):
        obj = BUILD / f"{src.stem}.o"
        res = subprocess.run([hipcc, *flags, "-c", str(src), "-o", str(obj)], capture_output=True, text=True, timeout=600)
        assert res.returncode == 0, res.stderr[-4000:]
        return str(obj)

    with ThreadPoolExecutor(4) as pool:
        objs = list(pool.map(one, sources))
    # the device code's images are left out
    res = subprocess.run([hipcc, "-Xarch_host", "-fsanitize=address", "-Wl,--unresolved-symbols=ignore-all", *objs, "-o", str(exe)],
                         capture_output=True, text=True, timeout=600)
    assert res.returncode == 0, res.stderr[-4000:]
    return exe


def check(driver, name, **env):
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0:abort_on_error=1", **env)
    env.pop("FULLWAVE_HIP_KERNELS", None)
    res = subprocess.run([str(driver), name], capture_output=True, text=True, timeout=300, env=env)
    print(res.stdout[-2000:], res.stderr[-6000:])
    assert res.returncode == 0
    assert f"{name}: ok" in res.stdout


def test_adjoint_on_a_handle_with_a_captured_graph(driver):
    check(driver, "graph_then_adjoint")


def test_kernels_of_a_handle_without_steps(driver):
    check(driver, "no_records")


def test_captured_steps_of_bricks_that_lose_their_codes(driver):
    check(driver, "graph_without_codes")


def test_kernels_of_bricks_that_lose_their_codes(driver):
    check(driver, "kernels_without_codes")


def test_timing_keeps_the_fastest_kernels(driver):
    check(driver, "timing")


def test_per_axis_maps_uploaded_again(driver):
    check(driver, "per_axis_uploads")


def test_adjoint_destroyed_before_and_after_its_simulation(driver):
    check(driver, "adjoint_lifetimes")


def test_kernels_of_taped_steps(driver):
    check(driver, "taped_kernels")
