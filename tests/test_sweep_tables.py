"""Packed sweep tables whose allocation fails leave nothing behind and are not
asked for again (tests/cpp/sweep_tables.cpp, on the host)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")
def test_allocation_failures(tmp_path):
    exe = tmp_path / "sweep_tables"
    subprocess.run([HIPCC, "-O0", "-std=c++17", "--offload-arch=gfx950", "-ffp-contract=off", "-Xclang",
                    "-target-feature", "-Xclang", "-packed-fp32-ops", "-w", "-I", os.path.join(ROOT, "include"), "-I",
                    os.path.join(ROOT, "unap_amd", "csrc"), os.path.join(ROOT, "tests", "cpp", "sweep_tables.cpp"),
                    "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
