"""The host-buffer transfers of a context (csrc/staging.h) on a stand-in HIP runtime whose stream runs only where it
is waited for: no GPU. No counterpart in the reference, which copies with the backend's own tensor calls."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("staging") / "host_staging")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I" + os.path.join(ROOT, "jepa.cpp_amd", "csrc"),
                    os.path.join(ROOT, "tests", "host_staging.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("case", [
    "slots",       # transfers of one to many pieces: no slot is filled again or read before its copy is done
    "refused",     # no pinned memory: the same transfers through the runtime's copies, and no error left on the thread
    "direct",      # uploads of more than one slot, and from memory the runtime knows, are one copy from where it is
    "stale",       # an error that an earlier call left on the thread does not refuse a transfer; a failed launch does
])
def test_staging(program, case):
    r = subprocess.run([program, case], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
