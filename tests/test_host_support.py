"""Host-side support of the kernel launchers, by a native driver (tests/native/host_support.cc) under the address and
undefined-behaviour sanitizers.  Host code only."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM_INCLUDE = "/opt/rocm/include"
READELF = "/opt/rocm/llvm/bin/llvm-readelf"


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


def _kernel_metadata(library, tmp_path):
    """(mangled name, VGPRs spilled, scratch bytes a lane) of every kernel in a library that was built here."""
    data, found, at = open(library, "rb").read(), [], 1
    while (at := data.find(b"\x7fELF", at)) >= 0:
        if data[at + 18:at + 20] == b"\xe0\x00":  # EM_AMDGPU
            code = tmp_path / "code.elf"
            code.write_bytes(data[at:])  # the header says where it ends
            notes = subprocess.run([READELF, "--notes", str(code)], capture_output=True, text=True, timeout=120).stdout
            for kernel in notes.split(".agpr_count:")[1:]:
                field = lambda key: re.search(r"\." + key + r":\s+(\S+)", kernel).group(1)
                found.append((field("symbol"), int(field("vgpr_spill_count")), int(field("private_segment_fixed_size"))))
        at += 4
    return found


def test_generic_kernels_without_rotation_hold_their_operands_in_registers(tmp_path):
    """The generic attention kernels of plain caches, alone and two in a launch, spill nothing (those that rotate inside do)."""
    library = os.path.join(ROOT, "tvm_amd", "lib", "libtvmkv.so")
    if not (os.path.exists(READELF) and os.path.exists(library)):
        pytest.skip("needs the built library and llvm-readelf")
    plain = [k for k in _kernel_metadata(library, tmp_path)
             if "generic_pair_kernel" in k[0] or re.search(r"generic_attn_kernelI.*ELb0EE", k[0])]
    assert len(plain) == 14  # 2 storage types x 5 tiles, 2 x 2 pairs
    assert [k for k in plain if k[1] or k[2]] == []


def test_prefill_kernels_of_head_dim_256_keep_no_copy_addresses(tmp_path):
    """The plain ragged and paged forms spill 8 and 10 registers at most; with the addresses of a tile's copies among the
    values that are kept from tile to tile it was 14 and 16, and their reloads waited for the copies in flight."""
    library = os.path.join(ROOT, "tvm_amd", "lib", "libtvmkv.so")
    if not (os.path.exists(READELF) and os.path.exists(library)):
        pytest.skip("needs the built library and llvm-readelf")
    plain = [k for k in _kernel_metadata(library, tmp_path) if re.search(r"prefill_kernelILi256ELi256ELi[01]ELi16ELb0E", k[0])]
    assert len(plain) == 3
    assert [k for k in plain if k[1] > 10] == []
