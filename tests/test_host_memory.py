"""Device buffers, their pool and host copies (pssa_amd/csrc/common.h) on the
CPU: tests/host_memory.cpp, built with the runtime's memory calls replaced by a
heap of a fixed size, so that running out of memory needs no GPU."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT
from pssa_amd.build import HIPCC


def test_buffers_pool_and_host_copies(tmp_path):
    if shutil.which(HIPCC) is None:
        pytest.skip("no hipcc")
    obj, exe = str(tmp_path / "t.o"), str(tmp_path / "t")
    subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-O1", "-std=c++17", "-fPIC", "-w", "-c",
                    os.path.join(ROOT, "tests", "host_memory.cpp"), "-o", obj], check=True)
    subprocess.run(["g++", obj, "-o", exe, "-lpthread"], check=True)
    run = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0, run.stdout
