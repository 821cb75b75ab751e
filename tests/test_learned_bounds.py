"""Every address that the learned preconditioner's kernels touch lies inside its
buffer: the kernels run on the CPU (host_hip/hip/hip_runtime.h), where an access
past the end of an allocation is a segmentation fault.  Panels with an odd side
have a number of edges that is no multiple of four, so that a launch of 64
threads per edge in blocks of 256 ends with threads that have no edge; 15 x 15
with six pairs is the shape at which a training gradient once faulted on the
GPU."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CLANG = "/opt/rocm/llvm/bin/clang++"


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("bounds") / "learned_bounds")
    subprocess.run([CLANG, "-std=c++17", "-O2", "-w", "-pthread", "-I", os.path.join(HERE, "host_hip"), "-x", "c++",
                    os.path.join(HERE, "learned_bounds.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.skipif(not os.path.exists(CLANG), reason="needs ROCm's clang++")
@pytest.mark.parametrize("args,edges", [((1, 1), 10), ((3, 2), 66), ((4, 2), 112), ((15, 6, 1), 1410)])
def test_kernels_stay_inside_their_buffers(program, args, edges):
    r = subprocess.run([program, *map(str, args)], capture_output=True, text=True, timeout=110)
    assert r.returncode == 0, (r.returncode, r.stdout)
    assert f" {edges} edges " in r.stdout
