"""Host code of the library on the CPU, as it is compiled for it, linked with stand-ins for the runtime
calls it makes: what moves host tensors (csrc/host_io.hip, host_io_check.cpp), what asks for LDS
(LdsGrant in csrc/plan.hpp, lds_grant_check.cpp) and a forward pass in one call (csrc/api.hip,
pass_stream_check.cpp); and the rows that the matrix-core kernels read (csrc/tap_walk.hpp,
tap_walk_check.cpp)."""
import os
import subprocess

import pytest

from xnor_nn_amd import build

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    """Builds a program of the given sources, host code only and without the HIP runtime."""
    try:
        hipcc = build.hipcc()
    except RuntimeError:
        pytest.skip("needs hipcc")
    at = tmp_path_factory.mktemp("host_code")
    built = {}

    def make(*sources):
        if sources not in built:
            objects = []
            for s in sources:
                objects.append(str(at / (os.path.basename(s) + ".o")))
                kind = ["-x", "hip", "--offload-arch=gfx950", "--offload-host-only",
                        "-fuse-cuid=" + ("none" if s.endswith(".hip") else "random")]
                subprocess.check_call([hipcc] + kind + [
                    "-O2", "-fPIC", "-std=c++17", "-I" + os.path.join(build.ROOT, "include"),
                    "-I" + build.SRC, "-c", s, "-o", objects[-1]])
            built[sources] = str(at / ("program%d" % len(built)))
            subprocess.check_call(["g++"] + objects + ["-o", built[sources], "-lpthread"])
        return built[sources]

    return make


def run(*command):
    out = subprocess.run(command, capture_output=True, text=True, timeout=100)
    assert out.returncode == 0 and out.stdout == "ok\n", (out.returncode, out.stdout, out.stderr)


@pytest.mark.parametrize("case", ["pinned tensors", "sizes", "bounded", "no pinned memory",
                                  "threads", "refused", "busy stream"])
def test_host_io(program, case):
    run(program(os.path.join(build.SRC, "host_io.hip"), os.path.join(HERE, "host_io_check.cpp")),
        case)


def test_lds_is_granted_to_two_threads(program):
    """Two threads that ask for different sizes: the larger one stays granted."""
    run(program(os.path.join(HERE, "lds_grant_check.cpp")))


@pytest.mark.parametrize("case", ["one pass", "stage fusion off", "popcount kernel", "old weights"])
def test_a_pass_keeps_its_stream(program, case):
    """Two threads with a stream each on one descriptor: all of a pass goes to its own."""
    run(program(os.path.join(build.SRC, "api.hip"), os.path.join(HERE, "pass_stream_check.cpp")), case)


def test_kernel_taps_read_staged_rows(program):
    """Nothing is read past what a tile has staged, not behind the last tap either."""
    run(program(os.path.join(HERE, "tap_walk_check.cpp")))
