"""The one-kernel CG loop (cg_cluster.hip) on the CPU: its own source, built by
the host compiler, with its workgroups, waves and threads run in random order
and one wave held back (emu/cluster_emu.cpp). Every order has to reach the
loop's end with the same bits; no wait may be left without an answer."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

pytestmark = pytest.mark.skipif(not shutil.which("g++"), reason="g++ not available")


@pytest.fixture(scope="module")
def emulation(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("cluster") / "cluster_emu")
    # -fno-extern-tls-init: the dynamic LDS array is declared inside the kernel;
    # -U_FORTIFY_SOURCE: the threads' stacks are changed by longjmp
    cmd = ["g++", "-std=c++17", "-O1", "-ffp-contract=off", "-U_FORTIFY_SOURCE", "-fno-extern-tls-init", "-w",
           "-I", os.path.join(HERE, "emu", "host_hip"), "-I", os.path.join(ROOT, "panopaea_amd", "csrc"),
           "-I", os.path.join(ROOT, "include"), os.path.join(HERE, "emu", "cluster_emu.cpp"), "-o", exe, "-pthread"]
    b = subprocess.run(cmd, capture_output=True, text=True, timeout=600)
    assert b.returncode == 0, b.stderr[-4000:]
    return exe


def test_cluster_orders(emulation):
    r = subprocess.run([emulation], capture_output=True, text=True, timeout=900)
    assert r.returncode == 0, (r.stdout[-3000:], r.stderr[-3000:])
