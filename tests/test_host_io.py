"""What moves host tensors (xnor_nn_amd/csrc/host_io.hip), on the CPU: its host code as the library
compiles it, with stand-ins for the runtime calls (host_io_check.cpp)."""
import os
import shutil
import subprocess

import pytest

from xnor_nn_amd import build

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    try:
        hipcc = build.hipcc()
    except RuntimeError:
        pytest.skip("needs hipcc")
    rocm = os.path.dirname(os.path.dirname(os.path.realpath(shutil.which(hipcc) or hipcc)))
    at = tmp_path_factory.mktemp("host_io")
    include = ["-I" + os.path.join(build.ROOT, "include"), "-I" + build.SRC]
    flags = ["-O2", "-fPIC", "-std=c++17"] + include
    lib, check, out = (str(at / n) for n in ("host_io.o", "check.o", "check"))
    subprocess.check_call([hipcc, "-x", "hip", "--offload-arch=gfx950", "--offload-host-only",
                           "-fuse-cuid=none"] + flags
                          + ["-c", os.path.join(build.SRC, "host_io.hip"), "-o", lib])
    subprocess.check_call(["g++", "-D__HIP_PLATFORM_AMD__", "-Wno-unused-result"] + flags
                          + ["-I" + os.path.join(rocm, "include"), "-c",
                             os.path.join(HERE, "host_io_check.cpp"), "-o", check])
    subprocess.check_call(["g++", lib, check, "-o", out, "-lpthread"])
    return out


@pytest.mark.parametrize("case", ["pinned tensors", "sizes", "bounded", "no pinned memory",
                                  "threads", "refused", "busy stream"])
def test_host_io(program, case):
    out = subprocess.run([program, case], capture_output=True, text=True, timeout=100)
    assert out.returncode == 0 and out.stdout == "ok\n", (out.returncode, out.stdout, out.stderr)
