"""Host copies through pinned staging memory, the host part on the CPU.

tests/csrc/staging_check.cpp drives m3.c_amd/csrc/hip/m3_staging.h over a
stream that runs nothing until it is waited for, with every step failing in
turn: staging memory may be used again only when no queued copy can touch it
any more.
"""
import os
import subprocess

from conftest import ROOT


def test_staged_copy_steps(tmp_path):
    binary = str(tmp_path / "staging_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-Wall",
                    "-Wextra", "-Werror", "-fsanitize=address,undefined",
                    "-I", os.path.join(ROOT, "m3.c_amd", "csrc", "hip"),
                    os.path.join(ROOT, "tests", "csrc", "staging_check.cpp"),
                    "-o", binary], check=True)
    result = subprocess.run([binary], capture_output=True, text=True,
                            timeout=120)
    assert result.returncode == 0, result.stdout + result.stderr
    assert "failures 0" in result.stdout
