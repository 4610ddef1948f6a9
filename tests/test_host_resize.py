"""The resize launcher where the runtime refuses to raise a kernel's LDS limit (tests/host_resize_driver.cpp): the frame goes through the kernel that needs
no more than the default, and the refusal is not reported as the launch's error.  No GPU: the driver stands in for the runtime."""
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "realtime-vla_amd"))


def test_a_refused_lds_limit_leaves_no_error_behind(tmp_path):
    import build as rtvla_build
    hipcc = rtvla_build._hipcc()
    if shutil.which(hipcc) is None and not os.path.exists(hipcc):
        pytest.skip("hipcc not found")
    obj, exe = str(tmp_path / "transforms.o"), str(tmp_path / "host_resize_driver")
    src = os.path.join(rtvla_build.CSRC, "transforms.hip")
    for cmd in ([hipcc] + rtvla_build.FLAGS + rtvla_build.EXTRA["transforms.hip"] + ["-c", src, "-o", obj],
                ["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", os.path.join(ROOT, "tests", "host_resize_driver.cpp"), obj, "-o", exe],
                [exe]):
        r = subprocess.run(cmd, capture_output=True, text=True)
        assert r.returncode == 0, (r.stdout + r.stderr)[-2000:]
    assert "all checks passed" in r.stdout
