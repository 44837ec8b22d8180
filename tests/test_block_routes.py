"""The block copy's dispatch, checked on the CPU: tests/block_routes_check.cc
compiled against libkvx."""
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
import bench  # noqa: E402


def test_block_copy_kernels_and_lds(tmp_path):
    """Which kernel a gather or scatter runs and the LDS it reserves, on both
    sides of each line of the rule; and what the benchmark says its isolated
    launches run is what they run."""
    cxx = shutil.which("g++") or shutil.which("c++")
    libdir = os.path.join(ROOT, "tpu-sync_amd")
    if cxx is None or not os.path.exists(os.path.join(libdir, "libkvx.so")):
        pytest.skip("no C++ compiler or libkvx.so not built")
    exe = tmp_path / "block_routes_check"
    env = {k: v for k, v in os.environ.items() if k != "LD_PRELOAD"}
    r = subprocess.run([cxx, "-O1", "-std=c++17", "-Wall", "-Werror", "-D__HIP_PLATFORM_AMD__",
                        "-I/opt/rocm/include",
                        "-I", os.path.join(ROOT, "tpu-sync_amd", "csrc", "kernels"),
                        os.path.join(ROOT, "tests", "block_routes_check.cc"), "-o", str(exe),
                        "-L", libdir, "-lkvx", f"-Wl,-rpath,{libdir}"],
                       capture_output=True, text=True, env=env)
    assert r.returncode == 0, r.stdout + r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120, env=env)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "all checks passed" in r.stdout
    for name, (kernel, kib) in bench.ISOLATED_PIECES.items():
        assert f"benchmark {name}: {kernel}, {kib} KiB\n" in r.stdout
