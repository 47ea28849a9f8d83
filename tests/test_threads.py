"""Host work on threads (fvens_amd/csrc/threads.hpp): every piece runs once however many threads can
be had, and no failure to start one ends the process. The header is compiled into
tests/threads_harness.cpp with g++."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("threads") / "threads_harness")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I",
                    os.path.join(ROOT, "fvens_amd", "csrc"),
                    os.path.join(ROOT, "tests", "threads_harness.cpp"), "-o", exe], check=True)

    def run(*args):
        p = subprocess.run([exe] + [str(a) for a in args], capture_output=True, text=True)
        assert p.returncode == 0, (args, p.returncode, p.stderr)
        return p.stdout.split()
    return run


@pytest.mark.parametrize("n", [1, 2, 8])
def test_every_piece_runs_once(harness, n):
    assert harness(n, 0) == ["1"] * n


@pytest.mark.parametrize("refused", range(1, 12))
def test_no_memory_for_a_thread(harness, refused):
    """The first allocations are the call's own (refused: nothing runs), the others the threads':
    the pieces without one run on the calling thread."""
    out = harness(8, refused)
    assert out in (["1"] * 8, ["0"] * 8 + ["bad_alloc"]), out
    assert refused <= 2 or out == ["1"] * 8


def test_an_exception_comes_back_after_the_others(harness):
    assert harness(8, -5) == ["1"] * 8 + ["piece"]
