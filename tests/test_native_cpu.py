"""Host code of the library on a stand-in for the HIP runtime (tests/native): compiled with the host compiler, no
device.  Each case is a program of its own; a hang ends at its time limit."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

HERE = os.path.join(ROOT, "tests", "native")


@pytest.fixture(scope="session")
def native(tmp_path_factory):
    """Builds one of tests/native/*.cpp; kernels and launchers stay unresolved (the cases launch none)."""
    built = {}

    def build(name):
        if name not in built:
            if shutil.which("g++") is None or not os.path.isdir("/opt/rocm/include/hip"):
                pytest.skip("needs g++ and the HIP headers")
            exe = str(tmp_path_factory.mktemp("native") / name)
            cmd = ["g++", "-std=c++17", "-O1", "-g", "-ftrapv", "-x", "c++", "-D__HIP_PLATFORM_AMD__", "-pthread",
                   "-I/opt/rocm/include", "-I", os.path.join(ROOT, "include"),
                   "-I", os.path.join(ROOT, "pypatools_amd", "csrc"), os.path.join(HERE, name + ".cpp"), "-o", exe,
                   "-Wl,--unresolved-symbols=ignore-all"]
            res = subprocess.run(cmd, capture_output=True, text=True)
            assert res.returncode == 0, res.stderr[-4000:]
            built[name] = exe
        return built[name]
    return build


def run(exe, case):
    res = subprocess.run([exe, case], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, f"{case}: exit {res.returncode}\n{res.stderr}"


@pytest.mark.parametrize("case", ["reuse_waits", "double_free", "free_and_capture", "destroyed_stream", "other_allocations",
                                  "bound_and_release", "devices_apart"])
def test_device_blocks(native, case):
    run(native("test_blocks"), case)


def test_no_module_allocates_past_the_kept_blocks():
    """hipMalloc itself fails while freed blocks are kept that could serve the request."""
    csrc = os.path.join(ROOT, "pypatools_amd", "csrc")
    for name in sorted(os.listdir(csrc)):
        if name != "pp_host.hip":
            with open(os.path.join(csrc, name)) as f:
                assert "hipMalloc(" not in f.read(), name
    with open(os.path.join(csrc, "pp_host.hip")) as f:
        blocks, rest = f.read().split("int ensure_init()", 1)
    assert "hipMalloc(" in blocks and "hipMalloc(" not in rest


@pytest.mark.parametrize("case", ["bytes", "no_error_left", "one_waiter", "devices_kept", "no_device_yet",
                                  "small_in_one_piece", "threads_by_size"])
def test_copies(native, case):
    run(native("test_copy"), case)


@pytest.mark.parametrize("case", ["gather", "node_index", "grids"])
def test_routes(native, case):
    run(native("test_routes"), case)


@pytest.mark.parametrize("case", ["pieces", "same_cell", "layout", "refused"])
def test_maps(native, case):
    run(native("test_maps"), case)
