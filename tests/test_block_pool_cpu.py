"""The bookkeeping of the kept device blocks (csrc/vkv_blockpool.h) over a host
allocator: counts, limits and lists while another thread waits for the device,
refused waits, a full device, and threads that release while others allocate;
and the library's device allocations on a device that is nearly full."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("pool") / "block_pool_check")
    # (assertions: an empty list's front() ends the program)
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-Wall", "-D_GLIBCXX_ASSERTIONS", "-pthread",
                    "-I", os.path.join(ROOT, "vmlx-swift_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "block_pool_check.cpp"), "-o", exe],
                   check=True)
    return exe


@pytest.mark.parametrize("case", ["release_during_wait", "give_and_take_during_wait",
                                  "refused_wait", "limits", "full_device", "threads"])
def test_block_pool(check, case):
    r = subprocess.run([check, case], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr


def test_scratch_on_a_full_device(tmp_path):
    """The library over a host allocator: where the device is full, a stream's
    scratch gets the memory of the kept blocks."""
    lib = os.path.join(ROOT, "vmlx-swift_amd")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    exe = str(tmp_path / "device_memory_check")
    # (exported: the library's HIP calls resolve to the program's functions)
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-Wall", "-rdynamic", "-I", f"{rocm}/include",
                    os.path.join(ROOT, "tests", "native", "device_memory_check.cpp"), "-o", exe,
                    f"-L{lib}", "-l:libvkv.so", f"-Wl,-rpath,{lib}", f"-L{rocm}/lib", "-lamdhip64",
                    f"-Wl,-rpath,{rocm}/lib"], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
