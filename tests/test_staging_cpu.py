"""Host copies through pinned staging memory, the host part on the CPU.

tests/csrc/staging_check.cpp drives m3.c_amd/csrc/hip/m3_staging.h over a
stream that runs nothing until it is waited for, with every step failing in
turn: staging memory may be used again only when no queued copy can touch it
any more. It also checks the memory's owner: one copy at a time per set, no
allocation while a set is free, a bound, and what closing handles frees.
Built with the address and with the thread sanitizer.
"""
import os
import subprocess

import pytest

from conftest import ROOT


@pytest.mark.parametrize("sanitizer", ["address,undefined", "thread"])
def test_staging(tmp_path, sanitizer):
    binary = str(tmp_path / "staging_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-Wall",
                    "-Wextra", "-Werror", "-fsanitize=" + sanitizer,
                    "-I", os.path.join(ROOT, "m3.c_amd", "csrc", "hip"),
                    os.path.join(ROOT, "tests", "csrc", "staging_check.cpp"),
                    "-o", binary], check=True)
    result = subprocess.run([binary], capture_output=True, text=True,
                            timeout=120)
    assert result.returncode == 0, result.stdout + result.stderr
    assert "failures 0" in result.stdout
