"""The library's host code around copies and waits, compiled with a stand-in for the HIP
runtime (``tests/host/fake_hip.hpp``): its failure paths need no device."""

import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not Path(HIPCC).exists(), reason="needs hipcc")
@pytest.mark.parametrize("name, said", [("transfer_check", "transfers ok"),
                                        ("wait_check", "waits ok")])
def test_host_code(name, said, tmp_path):
    exe = tmp_path / name
    subprocess.run([HIPCC, "--cuda-host-only", "-O1", "-std=c++17", "-nogpulib", "-pthread",
                    "-I", str(ROOT / "tests" / "host"), "-I", str(ROOT / "solprop_amd" / "csrc"),
                    str(ROOT / "tests" / "host" / f"{name}.cpp"), "-o", str(exe)], check=True)
    done = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert done.returncode == 0 and said in done.stdout, done.stdout + done.stderr
