"""The server's host blocks and copies (host_pool.hpp) and its fetch stage
(fetch_stage.hpp) on the CPU, under AddressSanitizer (emu/*_check.cpp)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.mark.skipif(not shutil.which("g++"), reason="g++ not available")
@pytest.mark.parametrize("name", ["host_pool_check", "fetch_stage_check"])
def test_host_pool(name, tmp_path):
    exe = str(tmp_path / name)
    b = subprocess.run(["g++", "-std=c++17", "-O1", "-fsanitize=address", "-I", os.path.join(ROOT, "panopaea_amd", "csrc"),
                        "-I", os.path.join(HERE, "emu", "host_hip"), os.path.join(HERE, "emu", name + ".cpp"), "-o", exe, "-pthread"],
                       capture_output=True, text=True, timeout=300)
    assert b.returncode == 0, b.stderr[-4000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, (r.stdout[-3000:], r.stderr[-3000:])
