"""The read-back's host side (csrc/host_copy.h) on the CPU: tests/emu/
host_copy_emu.cpp compiles it with g++ under ThreadSanitizer, with the HIP calls
replaced by plain memory, and reads arrays back from one thread and from several
threads at once, as a program may that takes a simulation's positions in one
thread and its velocities in another.  The threads are on another device than
the simulation's, as a thread is that has chosen none: the copies are made on the
simulation's, and the thread's is as before afterwards."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROCM = "/opt/rocm/include"


@pytest.fixture(scope="module")
def emulator(tmp_path_factory):
    if shutil.which("g++") is None or not os.path.isdir(os.path.join(ROCM, "hip")):
        pytest.skip("needs g++ and the HIP headers")
    exe = str(tmp_path_factory.mktemp("emu") / "host_copy_emu")
    subprocess.run(["g++", "-std=c++17", "-O2", "-g", "-fsanitize=thread", "-pthread", "-D__HIP_PLATFORM_AMD__",
                    "-I" + ROCM, os.path.join(HERE, "emu", "host_copy_emu.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("threads", [1, 3])
def test_read_back_from_threads(emulator, threads):
    done = subprocess.run([emulator, str(threads)], capture_output=True, text=True, timeout=300)
    if "unexpected memory mapping" in done.stderr:
        pytest.skip("ThreadSanitizer does not run with this kernel's address layout")
    assert done.returncode == 0, done.stderr
