"""The host's wait for results in pinned memory, over a stub stream
(tests/c/wait_host_check.cpp): work queued behind the awaited kernel is not
waited for."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


@pytest.mark.skipif(shutil.which("g++") is None or not Path("/opt/rocm/include/hip").exists(),
                    reason="g++ or the HIP headers absent")
def test_wait_ends_with_the_awaited_store(tmp_path):
    exe = tmp_path / "wait_host"
    for cmd in (["g++", "-std=c++17", "-O1", "-Wall", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                 f"-I{ROOT / 'include'}", f"-I{ROOT / 'massivemds_amd/csrc'}",
                 str(ROOT / "tests/c/wait_host_check.cpp"), "-lpthread", "-o", str(exe)], [str(exe)]):
        proc = subprocess.run(cmd, capture_output=True, text=True, timeout=120)
        assert proc.returncode == 0, proc.stdout + proc.stderr
