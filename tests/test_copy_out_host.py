"""Results on their way to the caller's memory (copyout.cpp), without a GPU: compiled against a stand-in for the
runtime whose stream runs every launch at once, as a device that is always ahead of the caller, or in a thread of
its own.  Destinations pinned and pageable in every order: each gets its bytes and nothing beside them is written, no
call fails, and what the runtime copies by itself does not go through the windows too.  A context's first large
copies pin little memory: the first touch of its pages is part of their time."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("copyout") / "copyout_stream")
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-Wall", "-pthread", "-D__HIP_PLATFORM_AMD__",
                           "-I/opt/rocm/include", os.path.join(HERE, "copyout_stream.cpp"),
                           os.path.join(HERE, "..", "clovers_amd", "csrc", "copyout.cpp"), "-o", out])
    return out


@pytest.mark.parametrize("stream", ["at-once", "thread"])
def test_every_destination_gets_its_bytes(program, stream):
    p = subprocess.run([program, stream], capture_output=True, text=True, timeout=120)
    assert p.returncode == 0 and "FAILED" not in p.stdout, p.stdout[-2000:] + p.stderr[-2000:]
