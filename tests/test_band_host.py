"""The band solver's kernels and host code on the CPU (band_host.cpp,
host_hip/hip/hip_runtime.h): null pointers and accesses past the end of a
buffer are segmentation faults there."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CLANG = "/opt/rocm/llvm/bin/clang++"
pytestmark = pytest.mark.skipif(not os.path.exists(CLANG), reason="needs ROCm's clang++")


@pytest.fixture(scope="module")
def band_host(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("band") / "band_host")
    subprocess.run([CLANG, "-std=c++17", "-O2", "-w", "-pthread", "-I", os.path.join(HERE, "host_hip"), "-x", "c++",
                    os.path.join(HERE, "band_host.cpp"), "-o", exe], check=True)

    def run(*args):
        r = subprocess.run([exe, *map(str, args)], capture_output=True, text=True, timeout=110)
        assert r.returncode == 0, (r.returncode, r.stdout)
        return r.stdout
    return run


def test_solve_without_a_factorization_is_refused(band_host):
    band_host("unfactored")


def test_factorization_recovers_from_each_failed_allocation(band_host):
    out = band_host("memory")
    assert "chain sweeps: 2 allocations" in out and "block sweeps: 5 allocations" in out


# (equations, half-bandwidth, XCDs, workgroups at once on each, launches
# numbered by count up to): the dispatch starts one launch's workgroups first
# on every other XCD, so that workgroups that wait for others in index order
# fill both XCDs and never end
@pytest.mark.parametrize("n,b,xcds,slots,counted", [(600, 200, 4, 2, 1024), (600, 200, 2, 3, 1024), (700, 40, 4, 2, 1024),
                                                    (1000, 640, 4, 3, 1024), (2600, 300, 8, 8, 16)])
def test_two_handles_at_once(band_host, n, b, xcds, slots, counted):
    out = band_host("pair", n, b, xcds, slots, counted)
    assert out.count("ended") == 6


# (equations, half-bandwidth): one to five tile rows, a ragged last block, full
# bands in one, two and three blocks, helpers
@pytest.mark.parametrize("n,b", [(40, 10), (128, 127), (300, 40), (310, 309), (330, 300), (400, 150), (600, 599), (1300, 600)])
def test_schedules_and_sweeps_agree(band_host, n, b):
    assert band_host("solve", n, b).count("backward error") == 6
