"""Host-side support of the kernel launchers, by a native driver (tests/native/host_support.cc) under the address and
undefined-behaviour sanitizers.  Host code only."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM_INCLUDE = "/opt/rocm/include"


def test_host_support(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None or not os.path.isdir(ROCM_INCLUDE):
        pytest.skip("needs g++ and the HIP headers")
    exe = str(tmp_path / "host_support")
    built = subprocess.run([gxx, "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover=undefined",
                            "-D__HIP_PLATFORM_AMD__", "-I" + ROCM_INCLUDE, os.path.join(ROOT, "tests", "native", "host_support.cc"),
                            "-o", exe, "-pthread"], capture_output=True, text=True, timeout=600)
    assert built.returncode == 0, built.stderr[-4000:]
    # the harness of this environment preloads a library of its own; the sanitizer runtime only insists on coming first
    env = dict(os.environ, ASAN_OPTIONS="verify_asan_link_order=0", UBSAN_OPTIONS="print_stacktrace=1")
    run = subprocess.run([exe], capture_output=True, text=True, timeout=120, env=env)
    assert run.returncode == 0, (run.stdout + run.stderr)[-4000:]
    assert "all checks passed" in run.stdout
