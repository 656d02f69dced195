"""The library's host side where memory is short (tests/native/memory_limits.cpp):
what the pools keep for isolated attention is given back to an allocation that
would otherwise fail, blocks in use are not, and every allocation is freed."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "pretrained-rstr_amd", "csrc")


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="no hipcc")
def test_kept_blocks_give_way(tmp_path):
    objects = []
    for src in (os.path.join(CSRC, "rstr_hip.cpp"), os.path.join(HERE, "native", "memory_limits.cpp")):
        objects.append(str(tmp_path / (os.path.basename(src) + ".o")))
        subprocess.run(["hipcc", "-x", "hip", "--offload-arch=gfx950", "--cuda-host-only", "-std=c++17", "-O1", "-w",
                        "-c", src, "-o", objects[-1]], check=True, capture_output=True, timeout=300)
    # the launches that the checks do not reach stay unresolved
    exe = str(tmp_path / "memory_limits")
    subprocess.run(["g++", "-no-pie", *objects, "-Wl,--unresolved-symbols=ignore-all", "-o", exe, "-lpthread"], check=True,
                   capture_output=True, timeout=120)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", (r.returncode, r.stdout, r.stderr)
