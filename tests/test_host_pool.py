"""The host pool's rules (host_pool.hpp) on a runtime that only counts
(host_stub): reuse, bounds, release on a failed allocation and with the last
handle, no lock over a waiting hipFree, no exception without host memory.
(CPU only.)"""
import os
import re
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SOURCE = os.path.join(HERE, "host_pool_cases.cpp")
CASES = re.findall(r'^static void (\w+)\(\)$', open(SOURCE).read(), re.M)


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("host_pool") / "cases")
    csrc = os.path.join(os.path.dirname(HERE), "eman2_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-Wall", "-pthread", "-I" + os.path.join(HERE, "host_stub"),
                    "-I" + csrc, SOURCE, "-o", out], check=True)
    return out


def test_every_case_is_listed(program):
    names = subprocess.run([program], capture_output=True, text=True, check=True).stdout.split()
    assert sorted(names) == sorted(CASES)


@pytest.mark.parametrize("case", CASES)
def test_rule(program, case):
    r = subprocess.run([program, case], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
