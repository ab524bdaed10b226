"""The device memory that contexts keep, on the CPU: alloc.cpp built against
a HIP runtime of a pretended card (alloc_host.cpp), plainly and under the
host's thread sanitizer."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIP = "/opt/rocm/include"


@pytest.mark.parametrize("flags", [["-O2"], ["-O1", "-g", "-fsanitize=thread"]], ids=["plain", "threads"])
def test_kept_memory(tmp_path, flags):
    if not os.path.exists(os.path.join(HIP, "hip", "hip_runtime.h")):
        pytest.skip("no HIP headers")
    exe = str(tmp_path / "alloc_host")
    b = subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I" + HIP, *flags, "-o", exe,
                        os.path.join(ROOT, "tests", "alloc_host.cpp"),
                        os.path.join(ROOT, "accelerating-tc_amd", "csrc", "alloc.cpp"), "-lpthread"],
                       capture_output=True, text=True)
    if b.returncode and "-ltsan" in b.stderr:
        pytest.skip("no thread sanitizer runtime")
    assert b.returncode == 0, b.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout[-2000:] + r.stderr[-3000:]
