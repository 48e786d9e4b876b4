"""The host side of the LDL preconditioner (csrc/ldl_host.cpp), on the CPU:
tests/ldl_check.cpp is built with it and run."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "xcalibre_tw.jl_amd", "csrc")


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("ldl") / "ldl_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-pthread", "-I", CSRC,
                    os.path.join(HERE, "ldl_check.cpp"), os.path.join(CSRC, "ldl_host.cpp"), "-o", exe], check=True)

    def run(*args):
        r = subprocess.run([exe, *map(str, args)], capture_output=True, text=True, timeout=100)
        print(r.stdout)
        return r

    return run


@pytest.mark.parametrize("nx,ny", [(20, 20), (160, 120)])
def test_a_failed_allocation_reaches_the_caller(checker, nx, ny):
    """One thread (small factors) and several: never the end of the process."""
    r = checker("alloc", nx, ny)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)


@pytest.mark.parametrize("nx,ny", [(9, 7), (70, 66), (310, 140)])
def test_block_solves_round_as_the_substitution_does(checker, nx, ny):
    """Growth of a range's inverse cuts the range: no less accurate than the
    substitution on indefinite matrices either."""
    r = checker("solve", nx, ny)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)
